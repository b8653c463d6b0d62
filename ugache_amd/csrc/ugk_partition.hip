// Classify + partition by source, fused mixed-source extraction, key dedup.
//
// classify: one kernel does what the reference spreads over a lookup kernel, a 64-bit radix sort, a
// boundary kernel and four stream synchronisations.  A block takes a tile of 1024 keys (4 per lane, loaded
// coalesced), looks each key up (wavefront-cooperative for the hash table), derives positions with a
// wavefront ballot + popcount prefix and a 16-entry cross-wave table in LDS, reserves its output ranges with
// ONE atomic per source, stages the compacted records in LDS and writes them out as contiguous, coalesced
// runs: hits grow from the front of idx[], misses from the back, so idx[] and the two counters describe the
// same (location-grouped) array the reference obtains by sorting.
#include <cstdlib>

#include <mutex>
#include <type_traits>

#include "ugk_internal.h"
#include "ugk_mix.cuh"
#include "ugk_table.cuh"

// Scratch of ugk_dedup_static, the one entry point that allocates nothing: a header (word 0 = the epoch tag of the last
// call), then the slot set and the per-occurrence ids that ugk_dedup_* take from their workspace argument.  Every GPU
// the library runs on holds its own copy until the process ends; host code reaches it through the address
// hipGetSymbolAddress returns for the current device, never through this name.
#define UGK_DEDUP_STATIC_HEADER 256
#define UGK_DEDUP_STATIC_WS_BYTES (((size_t)2 * UGK_DEDUP_STATIC_MAX_KEYS) * 10 + 64)
static __device__ __align__(256) unsigned char scratch[UGK_DEDUP_STATIC_HEADER + UGK_DEDUP_STATIC_WS_BYTES];

namespace ugk {
namespace {

// Keys per lane of a classify / dedup pass: four for batches whose 1024-key tiles give every compute unit a workgroup
// (fewer atomics on the shared counters), one for smaller batches, which would leave compute units idle otherwise.
constexpr int kItems = 4;
static inline int items_for(size_t n) { return n >= (size_t)cu_count() * kBlock * kItems ? kItems : 1; }

template <typename K, int KIND, int ITEMS>
__global__ __launch_bounds__(kBlock) void classify_kernel(ugk_table_t t, const K *__restrict__ keys, size_t n,
                                                          uint64_t host_rows, const uint32_t *__restrict__ dst_map,
                                                          ugk_idx_t *__restrict__ idx,
                                                          uint32_t *counts, uint32_t *next_counts, uint32_t *status,
                                                          uint32_t *host_mirror) {
  constexpr int TILE = kBlock * ITEMS;  // keys per workgroup pass, ITEMS per lane
  __shared__ uint2 stage[TILE];
  __shared__ uint32_t wave_tot[ITEMS][kWavesPerBlock][2];
  __shared__ uint32_t base[2];
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1), wave = tid / kWave;
  const uint64_t lt_mask = (1ull << lane) - 1ull;

  if (blockIdx.x == 0 && tid == 0 && next_counts) {
    next_counts[0] = 0;
    next_counts[1] = 0;
  }

  for (size_t tile0 = (size_t)blockIdx.x * TILE; tile0 < n; tile0 += (size_t)gridDim.x * TILE) {
    uint32_t cls[ITEMS], off[ITEMS], pre[ITEMS];
    uint64_t key_of[ITEMS];
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      const size_t i = tile0 + (size_t)j * kBlock + tid;
      key_of[j] = i < n ? key_to_u64<K>(keys[i]) : 0;
    }
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      const size_t i = tile0 + (size_t)j * kBlock + tid;
      const bool active = i < n;
      const uint64_t key = key_of[j];
      const Found f = table_lookup<KIND>(t, key, active);
      uint32_t c = 0, o = 0;
      if (active) {
        if (f.hit && f.loc == UGK_LOC_LOCAL) {
          c = 1;
          o = f.off;
        } else if (f.hit && f.loc == UGK_LOC_HOST && f.off < host_rows) {
          c = 2;
          o = f.off;
        } else if (!f.hit && fallback_row(t, key) < host_rows && fallback_row(t, key) <= 0xffffffffull) {
          c = 2;
          o = (uint32_t)fallback_row(t, key);
        } else {
          atomicOr(status, UGK_ST_KEY_OUT_OF_RANGE);
          if (host_mirror) host_mirror[0] = UGK_ST_KEY_OUT_OF_RANGE;
        }
      }
      const uint64_t hb = __ballot(c == 1), mb = __ballot(c == 2);
      cls[j] = c;
      off[j] = o;
      pre[j] = (c == 1) ? __popcll(hb & lt_mask) : __popcll(mb & lt_mask);
      if (lane == 0) {
        wave_tot[j][wave][0] = __popcll(hb);
        wave_tot[j][wave][1] = __popcll(mb);
      }
    }
    __syncthreads();
    uint32_t H = 0, M = 0, hoff[ITEMS], moff[ITEMS];
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
#pragma unroll
      for (int w = 0; w < kWavesPerBlock; ++w) {
        if (w == wave) {
          hoff[j] = H;
          moff[j] = M;
        }
        H += wave_tot[j][w][0];
        M += wave_tot[j][w][1];
      }
    }
    if (tid == 0) {
      // both reservations with one 64-bit add (the two counters share an aligned word, neither can carry: their sum
      // stays below 2^32): atomics on one address are performed one after the other, so half as many is half the queue
      const unsigned long long add = ((unsigned long long)M << 32) | H;
      const unsigned long long before =
          add ? atomicAdd(reinterpret_cast<unsigned long long *>(counts), add) : 0ull;
      base[0] = (uint32_t)before;
      base[1] = (uint32_t)(before >> 32);
    }
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      uint32_t i32 = (uint32_t)(tile0 + (size_t)j * kBlock + tid);
      if (dst_map && cls[j] != 0) i32 = dst_map[i32];
      if (cls[j] == 1) stage[hoff[j] + pre[j]] = make_uint2(i32, off[j]);
      if (cls[j] == 2) stage[TILE - M + moff[j] + pre[j]] = make_uint2(i32, off[j]);
    }
    __syncthreads();
    uint2 *out = reinterpret_cast<uint2 *>(idx);
    const size_t hit0 = base[0];
    const size_t miss0 = n - (size_t)base[1] - M;
    for (uint32_t p = tid; p < H; p += kBlock) out[hit0 + p] = stage[p];
    for (uint32_t q = tid; q < M; q += kBlock) out[miss0 + q] = stage[TILE - M + q];
    __syncthreads();
  }
}

// ---- which keys are NOT served by the cache: one bit per key, a wavefront's ballot is one bitmap word ---------
template <typename K, int KIND>
__global__ __launch_bounds__(kBlock) void nonlocal_flags_kernel(ugk_table_t t, const K *__restrict__ keys, size_t n,
                                                                unsigned long long *__restrict__ flags) {
  const size_t n_words = (n + kWave - 1) / kWave;
  const int lane = (int)lane_id();
  for (size_t w = (size_t)blockIdx.x * kWavesPerBlock + threadIdx.x / kWave; w < n_words;
       w += (size_t)gridDim.x * kWavesPerBlock) {
    const size_t i = w * kWave + lane;
    const bool active = i < n;
    const uint64_t key = active ? key_to_u64<K>(keys[i]) : 0;
    const Found f = table_lookup<KIND>(t, key, active);
    const uint64_t bits = __ballot(active && !(f.hit && f.loc == UGK_LOC_LOCAL));
    if (lane == 0) flags[w] = bits;
  }
}

template <typename K>
__global__ __launch_bounds__(kBlock) void select_keys_kernel(const K *__restrict__ keys, const uint32_t *__restrict__ sel,
                                                             size_t m, K *__restrict__ out) {
  for (size_t j = (size_t)blockIdx.x * kBlock + threadIdx.x; j < m; j += (size_t)gridDim.x * kBlock)
    out[j] = keys[sel[j]];
}

// ---- fused lookup + gather: every wavefront resolves its keys, then copies their rows -----------------------
// Measured and dropped: persistent wavefronts over a flat table that work two batches ahead (while the rows of batch i
// are copied, the table words of batch i + 1 and the keys of batch i + 2 are on their way), on 2 - 16 workgroups per
// compute unit: bit-exact, and 1 - 8 % slower at every size (262,144 keys of 512 bytes, 1 % misses: 49.8 - 52.4 us
// against 48.5 us).  With eight short wavefronts per SIMD the chip already overlaps one wavefront's table round trip
// with the others' row copies, and wavefronts that stride over the batch give up the moving window of output rows
// that workgroups started in order write.
// the rows of one wavefront's KPW keys, lane l holding the address of key b0 + l's row, ROWS of them on their way per lane
// stage_bits (STAGE only): where the lane's row is filed as well, 0 for a row that is not
template <int LPR, int KPW, int ROWS, Store STORE, bool KEEP, bool STAGE>
__device__ __forceinline__ void mix_copy(const MixRow &row, uint64_t stage_bits, u32x4 *out, size_t b0, uint32_t vpr) {
  constexpr int RPW = kWave / LPR;  // rows per wavefront instruction
  constexpr int UNROLL = RPW * ROWS <= KPW ? ROWS : KPW / RPW;
  static_assert(KPW <= kWave && KPW % (RPW * UNROLL) == 0, "keys per wavefront must be whole rounds of rows");
  const int lane = (int)lane_id();
  const int sub = lane % LPR, rg = lane / LPR;
  for (int r0 = 0; r0 < KPW; r0 += RPW * UNROLL) {
    // the row addresses travel between lanes as integers; turned back into pointers they must be told to be global
    // memory again, or the loads become generic ones, which the hardware cannot keep several of in flight in order
    grow_t p[UNROLL];
    gout_t ps[UNROLL];
    bool ok[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      p[u] = reinterpret_cast<grow_t>(shfl64(row.bits, r0 + u * RPW + rg));
      ok[u] = __shfl((int)row.has_row, r0 + u * RPW + rg) != 0;
      if constexpr (STAGE) ps[u] = reinterpret_cast<gout_t>(shfl64(stage_bits, r0 + u * RPW + rg));
    }
    for (uint32_t c0 = 0; c0 < vpr; c0 += LPR) {
      const uint32_t col = c0 + sub;
      if (col < vpr) {
        u32x4 v[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
          if constexpr (KEEP) v[u] = p[u][col];
          else v[u] = __builtin_nontemporal_load(p[u] + col);
        }
        arrived(v);
        const gout_t dst = (gout_t)out + (b0 + r0 + rg) * vpr + col;
#pragma unroll
        for (int u = 0; u < UNROLL; ++u)
          if (ok[u]) {
            const gout_t to = dst + (size_t)u * RPW * vpr;
            if constexpr (STORE == kThrough) store_through(reinterpret_cast<uint64_t>(to), v[u]);
            else if constexpr (STORE == kStreaming) __builtin_nontemporal_store(v[u], to);
            else *to = v[u];
          }
        if constexpr (STAGE) {
#pragma unroll
          for (int u = 0; u < UNROLL; ++u)
            if (ps[u]) {
              if constexpr (STORE == kThrough) store_through(reinterpret_cast<uint64_t>(ps[u] + col), v[u]);
              else ps[u][col] = v[u];
            }
        }
      }
    }
  }
}

// A row taken from the host table is also filed in the stage (ugk_stage_t): entry h = fmix64(row) & mask.  The first
// wavefront of a launch that finds the entry not yet written by this launch, and not holding this very row already,
// claims it with one compare-and-swap on its owner word and writes the row's bytes next to its stores into the output;
// everybody else leaves it alone.  After the launch an owner word names the row whose bytes the entry holds.
__device__ __forceinline__ uint64_t stage_claim(const ugk_stage_t &stage, const MixRow &row, uint32_t vpr) {
  if (row.host_row > 0xffffffffull) return 0;
  const uint32_t r32 = (uint32_t)row.host_row;
  const uint64_t h = fmix64(row.host_row) & stage.mask;
  unsigned long long *owner = reinterpret_cast<unsigned long long *>(stage.owner_dev) + h;
  const unsigned long long cur = __atomic_load_n(owner, __ATOMIC_RELAXED);
  const uint32_t tag = (uint32_t)(cur >> 32);
  if (tag == stage.epoch || (tag != 0 && (uint32_t)cur == r32)) return 0;
  const unsigned long long want = ((unsigned long long)stage.epoch << 32) | r32;
  if (atomicCAS(owner, cur, want) != cur) return 0;
  return reinterpret_cast<uint64_t>(reinterpret_cast<u32x4 *>(stage.rows_dev) + h * vpr);
}

// Rows of 512 bytes and more of a wavefront with few keys: eight per lane on their way, half the rounds to memory of four.  us,
// launch to end of poll, four / eight, a hash table, all rows in HBM and a twentieth over the link: 1 KB x 512 13.1 / 12.5 and
// 14.8 / 14.1, x 16,384 19.5 / 18.3 and 29.2 / 28.9; 4 KB x 16 14.5 / 12.9 and 16.6 / 14.5, x 1,024 18.3 / 17.0 and 23.2 / 21.1; 512
// bytes x 16,384 16.6 / 15.5 and 21.3 / 21.1.  Behind a flat table, which is soon looked up in, a launch that fills the chip has
// enough of them on their way: 1 KB x 2,048 11.9 / 11.6 and 13.3 / 12.7, x 8,192 13.3 / 13.6 and 18.1 / 18.5; 4 KB x 1,024 16.3 / 15.3
// and 21.4 / 19.1, x 4,096 18.6 / 17.7 and 26.1 / 26.5, x 16,384 31.7 / 34.2: up to 4,096 keys there.  Behind a hash table up to the
// 65,536 of the first arm of the rule that gives 16 keys (512 bytes x 32,768 20.3 / 19.8, x 65,536 24.3 / 24.5; 2 KB x 16,384 24.8 / 24.0),
// not beyond 262,144, where they are 16 again (uniform keys and zipf 1.05, a five-hundredth over the link: 512 bytes x 400,000 77.4 /
// 77.9 and 64.9 / 66.3, x 524,000 111.6 / 112.1 and 79.9 / 82.2; with streaming stores, x 1,040,000, 199.8 / 200.7 and 187.5 / 184.6; 1 KB x
// 520,000 204.7 / 205.6 and 178.0 / 174.4).
constexpr int mix_rows(int lpr, int kpw) { return lpr >= 32 && kpw <= 16 && kWave / lpr * 8 <= kpw ? 8 : 4; }

// KEEP: rows are loaded the ordinary way instead of past the caches, where the keys that repeat find them.  Stores that are written
// through need no room there, and a table that is cached in part is one whose keys are skewed: uniform ones pay 1 to 2 % for what
// zipf 1.2 gains 5 to 25 % by.  us, launch to end of poll, past / kept, keys that were not looked up before, a five-hundredth of the
// rows over the link, uniform, zipf 0.8, 1.05 and 1.2: 512 bytes x 128 11.1 / 11.2, 10.8 / 10.8, 10.6 / 10.4 and 10.5 / 10.3; x 4,096 13.6 /
// 13.9, 13.3 / 13.4, 12.8 / 12.8 and 12.6 / 12.5; x 32,768 18.6 / 19.0, 18.0 / 18.3, 17.1 / 17.0 and 16.8 / 15.8; x 65,536 23.6 / 23.8, 22.6 /
// 22.8, 21.3 / 21.6 and 21.7 / 18.5; x 131,072 32.8 / 33.0, 31.5 / 31.1, 29.3 / 31.0 and 30.6 / 25.0; 1204 bytes x 27,869 25.5 / 25.8, 24.4 /
// 24.6, 23.5 / 23.9 and 23.8 / 19.6; 100 bytes x 20,971 16.4 / 16.8, 16.0 / 16.1, 15.0 / 15.3 and 14.8 / 14.8, x 671,088 60.8 / 64.0, 58.1 /
// 56.6, 51.5 / 50.0 and 48.9 / 44.6.  With a fiftieth over the link, which then bounds the launch, 1 % either way.  Beyond 64 MB rows
// of more than 64 bytes lose (512 bytes x 262,144 53.5 / 54.6, 51.0 / 50.6, 46.4 / 50.1 and 49.0 / 46.4; 100 bytes x 1,342,177 112 / 127 and
// 101 / 104); shorter ones, of which a line holds several, go on (64 bytes x 2,097,152 117 / 123, 107.5 / 107.9, 92.1 / 89.9 and 87.0 /
// 81.0).  Distinct keys repeat nothing within a launch; what the launch before has kept of the same rows makes them even (512
// bytes, 0.25 to 134 MB, uniform and zipf 1.2, 0.99 to 1.02 times as fast).
// LPR: lanes per row, or 0 for rows that are copied flat (flat_copy; f.tile rows at a time)
template <typename K, int KIND, int LPR, int KPW, int ROWS, Store STORE, bool KEEP, bool STAGE>
__global__ __launch_bounds__(kBlock) void extract_mix_kernel(ugk_table_t t, const K *__restrict__ keys, size_t n,
                                                             const void *__restrict__ cache, uint64_t cache_rows,
                                                             const void *__restrict__ host, uint64_t host_rows,
                                                             void *__restrict__ out, FlatRow f_row,
                                                             uint32_t *status, uint32_t *host_mirror,
                                                             Ending<STORE> done, ugk_stage_t stage) {
  __shared__ uint32_t block_tot[2];
  if (threadIdx.x < 2) block_tot[threadIdx.x] = 0;
  __syncthreads();
  n = launch_count(done, n);
  uint32_t wave_local = 0, wave_host = 0;  // rows this wavefront took from each source (wavefront-uniform)
  const int lane = (int)lane_id();
  const size_t wave_global = (size_t)blockIdx.x * kWavesPerBlock + threadIdx.x / kWave;
  const size_t n_waves = (size_t)gridDim.x * kWavesPerBlock;
  for (size_t b0 = wave_global * KPW; b0 < n; b0 += n_waves * KPW) {
    const size_t i = b0 + lane;
    const bool active = lane < KPW && i < n;
    const uint64_t key = active ? key_to_u64<K>(keys[i]) : 0;
    // a full wavefront of keys probes its eight home lines in one go (see hash_probe_home)
    // (fewer keys: their home lines in one go as well, and only the rounds of the probe that have keys to serve)
    constexpr int ROUNDS = KPW >= 8 ? KPW / 8 : 1;
    const Found f = table_lookup<KIND, (KPW == kWave || ROUNDS < 8) ? 1 : 2, ROUNDS>(t, key, active);
    typedef typename std::conditional<LPR == 0, char, u32x4>::type unit_t;
    const MixRow row = mix_resolve(t, key, active, f, static_cast<const unit_t *>(cache), cache_rows,
                                   static_cast<const unit_t *>(host), host_rows, out,
                                   LPR == 0 ? f_row.row_bytes : f_row.chunks, status, host_mirror);
    if (done.words) {
      // rows from the cache, and all others (host rows, and rows skipped for a key without a row: the launch is
      // flagged then and its group sizes mean nothing, but the two sums still add up to n)
      wave_local += __popcll(__ballot(row.from_cache));
      wave_host += __popcll(__ballot(active && !row.from_cache));
    }
    if constexpr (LPR == 0) {
      const uint64_t bits = row.has_row ? row.bits : row.bits | kNoRowBit;
      const uint32_t here = (uint32_t)min((size_t)KPW, n - b0);
      for (uint32_t r0 = 0; r0 < here; r0 += f_row.tile)
        flat_copy<true, STORE == kThrough, KEEP, true>(bits, 0, static_cast<char *>(out), b0, r0, min(f_row.tile, here - r0), f_row);
    } else {
      const uint32_t vpr = f_row.chunks;
      uint64_t stage_bits = 0;
      if constexpr (STAGE) stage_bits = stage_claim(stage, row, vpr);
      mix_copy<LPR, KPW, ROWS, STORE, KEEP, STAGE>(row, stage_bits, static_cast<u32x4 *>(out), b0, vpr);
    }
    // behind the rows: in front of them it would be in the way of the lookup
    if constexpr (STORE == kThrough) {
      if (active) copy_key_along<K>(done, i, (K)key);
    }
  }
  if (done.words) mix_leave_counts(block_tot, wave_local, wave_host, done);
}

// ---- dedup -----------------------------------------------------------------------------------------------
// slot word = (epoch << 32) | index of the first occurrence that claimed the slot.  A slot whose epoch is not
// the current one is free, so the set never needs clearing between batches.
template <typename K, int ITEMS>
__global__ __launch_bounds__(kBlock) void dedup_claim_kernel(const K *__restrict__ keys, size_t n,
                                                             unsigned long long *slots, size_t cap_mask,
                                                             uint32_t epoch, const uint32_t *epoch_dev,
                                                             uint32_t *uid_of, K *unique_out, uint32_t *inverse,
                                                             uint32_t *rep_of, uint32_t *n_unique) {
  if (epoch_dev) epoch = *epoch_dev;  // the tag lives in device memory when the set does (see ugk_dedup_static)
  // A tile of TILE keys per pass (ITEMS per lane): one reservation of unique ids per tile, so with four per lane the
  // single counter they come from sees a quarter of the atomics a 256-key tile would send it.
  // Two stages.  The keys of a tile first meet in a set in LDS, where every distinct key of the tile gets one leader
  // (the occurrence whose claim came first); only leaders go on to the device-wide set.  Claims on one slot are
  // performed one after the other, in LDS within tens of nanoseconds, in device memory a round trip to the memory side
  // each: without the first stage a batch of skewed keys queues up on the slots of its hot keys (1 M keys, Zipf 1.1:
  // three times the time of 1 M distinct keys; all keys equal: twenty times).
  constexpr int TILE = kBlock * ITEMS;
  constexpr uint32_t LCAP = 2 * TILE;  // local set, at most half full
  constexpr uint32_t kNone = 0xffffffffu;
  __shared__ uint32_t wave_tot[ITEMS][kWavesPerBlock];
  __shared__ uint32_t base;
  __shared__ K skey[TILE];          // the tile's keys, by position in the tile
  __shared__ uint32_t lset[LCAP];   // local set: position of the leader that claimed the slot
  __shared__ uint32_t srep[TILE];   // leaders: index (in the batch) of their key's representative
  __shared__ K stage[TILE];
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1), wave = tid / kWave;
  for (size_t tile0 = (size_t)blockIdx.x * TILE; tile0 < n; tile0 += (size_t)gridDim.x * TILE) {
    bool winner[ITEMS];
    K key[ITEMS];
    uint32_t pre[ITEMS], leader[ITEMS];
    for (uint32_t q = tid; q < LCAP; q += kBlock) lset[q] = kNone;
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      const size_t i = tile0 + (size_t)j * kBlock + tid;
      key[j] = i < n ? keys[i] : K(0);
      skey[j * kBlock + tid] = key[j];
    }
    __syncthreads();
    // stage 1: one leader per distinct key of the tile
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      const size_t i = tile0 + (size_t)j * kBlock + tid;
      const uint32_t me = (uint32_t)(j * kBlock + tid);
      leader[j] = kNone;
      if (i < n) {
        uint32_t h = (uint32_t)(fmix64(key_to_u64<K>(key[j])) >> 32) & (LCAP - 1);
        for (;;) {
          uint32_t cur = lset[h];
          if (cur == kNone) cur = atomicCAS(&lset[h], kNone, me);
          if (cur == kNone) {
            leader[j] = me;
            break;
          }
          if (skey[cur] == key[j]) {
            leader[j] = cur;
            break;
          }
          h = (h + 1) & (LCAP - 1);
        }
      }
    }
    // stage 2: the leaders claim their keys in the device-wide set, one key of a lane after the other (sending a
    // lane's four first probes out together was slower: 1 M distinct keys 94 -> 142 us; the memory side performs the
    // claims no faster for being asked all at once)
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      const size_t i = tile0 + (size_t)j * kBlock + tid;
      const uint32_t me = (uint32_t)(j * kBlock + tid);
      winner[j] = false;
      if (i < n && leader[j] == me) {
        size_t h = fmix64(key_to_u64<K>(key[j])) & cap_mask;
        uint32_t rep = (uint32_t)i;
        for (;;) {
          unsigned long long s = __atomic_load_n(slots + h, __ATOMIC_RELAXED);
          bool claimed = false;
          while ((uint32_t)(s >> 32) != epoch) {
            const unsigned long long want = ((unsigned long long)epoch << 32) | (uint32_t)i;
            const unsigned long long seen = atomicCAS(slots + h, s, want);
            if (seen == s) {
              claimed = true;
              break;
            }
            s = seen;
          }
          if (claimed) {
            winner[j] = true;
            break;
          }
          const uint32_t other = (uint32_t)s;
          if (keys[other] == key[j]) {
            rep = other;
            break;
          }
          h = (h + 1) & cap_mask;
        }
        srep[me] = rep;
      }
      const uint64_t wb = __ballot(winner[j]);
      pre[j] = __popcll(wb & ((1ull << lane) - 1ull));
      if (lane == 0) wave_tot[j][wave] = __popcll(wb);
    }
    __syncthreads();
    uint32_t total = 0, before[ITEMS];
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
#pragma unroll
      for (int w = 0; w < kWavesPerBlock; ++w) {
        if (w == wave) before[j] = total;
        total += wave_tot[j][w];
      }
    }
    if (tid == 0) base = total ? atomicAdd(n_unique, total) : 0u;
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      const size_t i = tile0 + (size_t)j * kBlock + tid;
      if (winner[j]) stage[before[j] + pre[j]] = key[j];
      // index of the representative; replaced by its unique id in the second kernel
      if (i < n) inverse[i] = srep[leader[j]];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      if (winner[j]) {
        const size_t i = tile0 + (size_t)j * kBlock + tid;
        const uint32_t uid = base + before[j] + pre[j];
        uid_of[i] = uid;
        if (rep_of) rep_of[uid] = (uint32_t)i;
      }
    }
    for (uint32_t p = tid; p < total; p += kBlock) unique_out[base + p] = stage[p];
    __syncthreads();
  }
}

__global__ __launch_bounds__(kBlock) void dedup_resolve_kernel(size_t n, const uint32_t *__restrict__ uid_of,
                                                               uint32_t *inverse, const uint32_t *n_unique,
                                                               uint32_t *n_unique_host, uint32_t *next_n_unique) {
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (next_n_unique) *next_n_unique = 0;
    // (there before this launch has ended: the host may learn of that from the words of a launch behind this one, which an
    // ordinary store, acknowledged before it is in host memory, can be overtaken by)
    if (n_unique_host) tell_host(n_unique_host, *n_unique);
  }
  for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kBlock)
    inverse[i] = uid_of[inverse[i]];
}

// A batch that one workgroup holds, in one launch.  The two kernels above are a chain of round trips to the memory side, a slot read, a
// claim, the reservation of ids, and a second launch that follows the positions: 11 us and 4 for 3,321 keys, on a chip that is idle.
// Here all of it is in LDS: the keys, a set of them at most a quarter full, and in a claimed slot first the position that claimed
// it, then the id.  us per call, two kernels / this, uniform and zipf 1.2: 546 keys 8.3 / 5.0 and 8.7 / 5.0, 2,048 9.4 / 4.9 and 8.8 /
// 4.9, 4,096 10.1 / 7.2 and 8.8 / 5.8; a lookup of the distinct keys, rows of 512 bytes and their gather back by position, 546 keys
// 32.7 / 25.3, 2,000 34.7 / 26.9, 4,096 37.7 / 31.6.  Bound by the LDS of one CU from there on, with a set half full and 8,192 keys
// 11.2 / 17.4.  (A lane's four keys looking for their slots at the same time: 11.7 for 4,096 keys.)
constexpr int kSmallBlock = 1024;
constexpr size_t kSmallBatch = 4 * kSmallBlock;
template <typename K, int ITEMS>
__global__ __launch_bounds__(kSmallBlock) void dedup_small_kernel(const K *__restrict__ keys, uint32_t n, K *__restrict__ unique_out,
                                                                  uint32_t *__restrict__ inverse, uint32_t *__restrict__ rep_of,
                                                                  uint32_t *n_unique, uint32_t *n_unique_host,
                                                                  uint32_t *next_n_unique) {
  constexpr uint32_t kSlots = 4 * kSmallBlock * ITEMS, kNone = 0xffffffffu;
  constexpr int kWaves = kSmallBlock / kWave;
  __shared__ K skey[kSmallBlock * ITEMS];
  __shared__ uint32_t slots[kSlots];
  __shared__ uint32_t wave_tot[ITEMS][kWaves];
  const uint32_t tid = threadIdx.x, lane = lane_id(), wave = wave_in_block();
  K key[ITEMS];
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    const uint32_t i = (uint32_t)j * kSmallBlock + tid;
    key[j] = i < n ? keys[i] : K(0);
  }
  for (uint32_t q = tid; q < kSlots; q += kSmallBlock) slots[q] = kNone;
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) skey[(uint32_t)j * kSmallBlock + tid] = key[j];
  __syncthreads();
  uint32_t slot[ITEMS], pre[ITEMS];
  bool first[ITEMS];
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    const uint32_t i = (uint32_t)j * kSmallBlock + tid;
    uint32_t h = (uint32_t)(fmix64(key_to_u64<K>(key[j])) >> 32) & (kSlots - 1);
    first[j] = false;
    if (i < n) {
      for (;;) {
        uint32_t cur = slots[h];
        if (cur == kNone) cur = atomicCAS(&slots[h], kNone, i);
        if (cur == kNone) {
          first[j] = true;
          break;
        }
        if (skey[cur] == key[j]) break;
        h = (h + 1) & (kSlots - 1);
      }
    }
    slot[j] = h;
    const uint64_t mine = __ballot(first[j]);
    pre[j] = __popcll(mine & ((1ull << lane) - 1ull));
    if (lane == 0) wave_tot[j][wave] = __popcll(mine);
  }
  __syncthreads();
  uint32_t total = 0;
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      if (w == (int)wave) pre[j] += total;
      total += wave_tot[j][w];
    }
  }
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    if (first[j]) {
      slots[slot[j]] = pre[j];
      unique_out[pre[j]] = key[j];
      if (rep_of) rep_of[pre[j]] = (uint32_t)j * kSmallBlock + tid;
    }
  }
  if (tid == 0) {
    *n_unique = total;
    if (next_n_unique) *next_n_unique = 0;
    if (n_unique_host) tell_host(n_unique_host, total);  // as dedup_resolve_kernel does
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    const uint32_t i = (uint32_t)j * kSmallBlock + tid;
    if (i < n) inverse[i] = slots[slot[j]];
  }
}

// ugk_dedup_static, before the claims: when the epoch tag is about to wrap, every slot is cleared so that what was
// tagged 2^32 calls ago cannot read as current (the tag itself moves in static_epoch_kernel, after every workgroup of
// this kernel has read it)
__global__ __launch_bounds__(kBlock) void static_wrap_kernel(const uint32_t *epoch, unsigned long long *slots,
                                                             size_t cap) {
  if (*epoch != 0xffffffffu) return;
  for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < cap; i += (size_t)gridDim.x * kBlock) slots[i] = 0ull;
}

__global__ void static_epoch_kernel(uint32_t *epoch, uint32_t *n_unique, uint32_t *n_unique_host) {
  const uint32_t e = *epoch;
  *epoch = e == 0xffffffffu ? 1u : e + 1u;
  *n_unique = 0u;
  if (n_unique_host) *n_unique_host = 0u;  // an empty batch launches nothing else; a full one overwrites it
}

size_t dedup_capacity(size_t n) {
  size_t cap = 1024;
  while (cap < 2 * n) cap <<= 1;
  return cap;
}

template <typename K>
int classify(ugk_table_t t, const K *keys, size_t n, uint64_t host_rows, const uint32_t *dst_map, ugk_idx_t *idx,
             uint32_t *counts, uint32_t *next_counts, uint32_t *status, uint32_t *host_mirror, void *stream) {
  UGK_REQUIRE(counts && status, "ugk_classify: null counters or status");
  UGK_REQUIRE(n <= 0xffffffffull, "ugk_classify: batch of %zu keys exceeds 2^32", n);
  UGK_REQUIRE((uintptr_t)counts % 8 == 0, "ugk_classify: the two counters must share an 8-byte aligned word");
  UGK_REQUIRE(t.kind >= 1 && t.kind <= 3, "ugk_classify: table kind %d is not flat(1), hash(2) or compact hash(3)", t.kind);
  UGK_REQUIRE(t.table && t.size, "ugk_classify: empty table");
  if (t.kind >= 2)
    UGK_REQUIRE(t.size % (t.kind == 2 ? 8 : 16) == 0 && (uintptr_t)t.table % 128 == 0,
                "ugk_classify: hash table must be 128-byte aligned with whole 128-byte lines of buckets");
  UGK_REQUIRE(n == 0 || (keys && idx), "ugk_classify: null keys or index list");
  // n == 0 still launches one block so that next_counts is cleared
  const int items = items_for(n);
  const size_t tile = (size_t)kBlock * items;
  const unsigned grid = clamp_grid((n + tile - 1) / tile, 0);
#define UGK_GO(KIND, ITEMS)                                                                                       \
  hipLaunchKernelGGL((classify_kernel<K, KIND, ITEMS>), dim3(grid), dim3(kBlock), 0, as_stream(stream), t, keys, \
                     n, host_rows, dst_map, idx, counts, next_counts, status, host_mirror)
  if (t.kind == 1 && items == 1) UGK_GO(1, 1);
  else if (t.kind == 1) UGK_GO(1, kItems);
  else if (t.kind == 2 && items == 1) UGK_GO(2, 1);
  else if (t.kind == 2) UGK_GO(2, kItems);
  else if (items == 1) UGK_GO(3, 1);
  else UGK_GO(3, kItems);
#undef UGK_GO
  UGK_HIP(hipGetLastError());
  return 0;
}

template <typename K>
int nonlocal_flags(ugk_table_t t, const K *keys, size_t n, uint64_t *flags, void *stream) {
  if (n == 0) return 0;
  UGK_REQUIRE(keys && flags, "ugk_nonlocal_flags: null keys or bitmap");
  UGK_REQUIRE((uintptr_t)flags % 8 == 0, "ugk_nonlocal_flags: the bitmap must be 8-byte aligned");
  UGK_REQUIRE(t.kind >= 1 && t.kind <= 3, "ugk_nonlocal_flags: table kind %d is not flat(1), hash(2) or compact hash(3)", t.kind);
  UGK_REQUIRE(t.table && t.size, "ugk_nonlocal_flags: empty table");
  if (t.kind >= 2)
    UGK_REQUIRE(t.size % (t.kind == 2 ? 8 : 16) == 0 && (uintptr_t)t.table % 128 == 0,
                "ugk_nonlocal_flags: hash table must be 128-byte aligned with whole 128-byte lines of buckets");
  const unsigned grid = clamp_grid((n + kBlock - 1) / kBlock, 0);
  if (t.kind == 1)
    hipLaunchKernelGGL((nonlocal_flags_kernel<K, 1>), dim3(grid), dim3(kBlock), 0, as_stream(stream), t, keys, n,
                       reinterpret_cast<unsigned long long *>(flags));
  else if (t.kind == 2)
    hipLaunchKernelGGL((nonlocal_flags_kernel<K, 2>), dim3(grid), dim3(kBlock), 0, as_stream(stream), t, keys, n,
                       reinterpret_cast<unsigned long long *>(flags));
  else
    hipLaunchKernelGGL((nonlocal_flags_kernel<K, 3>), dim3(grid), dim3(kBlock), 0, as_stream(stream), t, keys, n,
                       reinterpret_cast<unsigned long long *>(flags));
  UGK_HIP(hipGetLastError());
  return 0;
}

template <typename K>
int select_keys(const K *keys, const uint32_t *sel, size_t m, K *out, void *stream) {
  if (m == 0) return 0;
  UGK_REQUIRE(keys && sel && out, "ugk_select_keys: null pointer");
  const unsigned grid = clamp_grid((m + kBlock - 1) / kBlock, 0);
  hipLaunchKernelGGL(select_keys_kernel<K>, dim3(grid), dim3(kBlock), 0, as_stream(stream), keys, sel, m, out);
  UGK_HIP(hipGetLastError());
  return 0;
}

template <typename K, int KIND>
int extract_mix_lpr(ugk_table_t t, const K *keys, size_t n, const void *cache, uint64_t cache_rows, const void *host,
                    uint64_t host_rows, void *out, size_t row_bytes, bool flat, uint32_t *status,
                    uint32_t *host_mirror, uint64_t *counts, uint32_t *num_groups, uint32_t others_hint, const ugk_stage_t *stage,
                    DoneRequest &request, hipStream_t st) {
  // ordinary write-back stores while the output fits the memory-side cache (the consumer finds it there),
  // non-temporal beyond, or as the caller's hint says
  const bool nt = !request.counted() && nt_store_for(n * row_bytes);
  const uint32_t vpr = (uint32_t)((row_bytes + 15) / 16);
  // Keys per wavefront.  A wavefront resolves its keys together and then copies their rows a few at a time; once its
  // first stores are out, every later load of the wavefront returns behind them, so wavefronts of one round of rows
  // (8 keys of 512 bytes) keep memory busier than long ones, and short ones also fill a chip that a small batch
  // would leave half empty.  What speaks for longer wavefronts is the lookup: a hash probe works on all 64 lanes at
  // once, and with small rows the lookups are a larger share of the work.  Measured on MI355X, 1 % misses, 8 / 16 / 32 /
  // 64 keys per wavefront, us per launch:
  //   flat, 512-byte rows:  8,192 keys 5.7 / 6.9 / 10.2 / 16.2;  65,536 keys 15.9 / 16.0 / 16.1 / 19.9;  262,144 keys
  //                         48.6 / 49.5 / 50.8 / 47.7;  1 M keys 189.7 / 191.4 / 202.7 / 203.7
  //   flat, 128-byte rows:  65,536 keys 8.2 / 7.7 / 7.6 / 8.5;  262,144 keys 21.0 / 21.8 / 19.5 / 20.1;  1 M keys 64.8 /
  //                         65.5 / 64.0 / 64.2
  //   hash, 512-byte rows:  8,192 keys 12.4 / 13.8 / 17.5 / 23.3;  65,536 keys 25.9 / 24.5 / 26.3 / 30.8;  131,072 keys
  //                         38.2 / 37.8 / 32.7 / 35.1;  262,144 keys 63.0 / 58.7 / 61.3 / 53.1;  1 M keys 215.3 / 211.4 /
  //                         219.3 / 226.4
  //   hash, 128-byte rows:  65,536 keys 22.0 / 18.9 / 18.7 / 19.9;  262,144 keys 49.0 / 37.0 / 31.2 / 28.9;  1 M keys
  //                         150.7 / 112.3 / 82.1 / 79.5
  // and the same order at 10 % misses, where the host link bounds the launch and the spread is 1-3 %.  The batch sizes
  // above are multiples of the chip's wavefront slots (256 CUs x 32 = 8,192), which is how the rule below states them.
  // others_hint does not enter the shape any more: since the row loads of a wavefront are in flight together, the mix
  // of sources no longer changes which shape wins.  It caps the grid instead when most rows come over the host link:
  // rows of 512 bytes and more cross it faster from 128 workgroups than from as many as the batch would fill (56.9
  // against 52.7 GB/s for uniformly random rows), and the few rows the cache serves do not miss the other workgroups.
  const bool mostly_host = others_hint != UGK_HINT_UNKNOWN && (size_t)others_hint * 2 >= n && vpr >= 32;
  const size_t slots = (size_t)cu_count() * 4 * 8;
  const int lpr = vpr <= 1 ? 1 : vpr <= 2 ? 2 : vpr <= 4 ? 4 : vpr <= 8 ? 8 : vpr <= 16 ? 16 : vpr <= 32 ? 32 : 64;
  const bool small_rows = lpr <= 8;  // rows of up to 128 bytes
  // of n keys whose number is in a device word, the distinct ones of a batch, any number may be there: half of them is a guess for
  // the shape (a skewed batch of 262,144 has 38,000, a uniform one all but 7,000)
  const size_t likely = request.counted() ? n / 2 : n;
  int kpw;
  if (KIND == 1) {
    kpw = small_rows ? 32 : 8;
  } else if (likely <= slots) {
    kpw = 8;
  } else if (small_rows) {
    kpw = likely <= slots * 16 ? 32 : 64;
  } else {
    kpw = likely <= slots * 8 ? 16 : likely <= slots * 16 ? 32 : likely <= slots * 32 ? 64 : 16;
  }
  // UGK_MIX_KPW=8|16|32|64 forces the shape (read on every launch: the sweep that measures the rule above changes it
  // between launches); never a byte of the result depends on it
  if (const char *forced = getenv("UGK_MIX_KPW")) {
    const int v = atoi(forced);
    if (v == 8 || v == 16 || v == 32 || v == 64) kpw = v;
  }
  if (!flat && kpw < kWave / lpr) kpw = kWave / lpr;  // one wavefront instruction copies 64 / lpr rows
  // a wavefront copies all its rows as one run of vectors, or a row at a time where they are too long to divide by
  const FlatRow f_row = flat_row(row_bytes, (uint32_t)kpw);
  const size_t keys_per_group = (size_t)kpw * kWavesPerBlock;
  const unsigned grid = request.grid(clamp_grid((n + keys_per_group - 1) / keys_per_group, mostly_host ? 128u : 0u));
  // Words come sooner than a ticket behind the launch would.  us, launch to end of poll, ticket / words, keys that were not looked up
  // before, uniform, a five-hundredth over the link, a hash table: 512 bytes x 1 11.7 / 9.7, x 1,024 14.6 / 13.4, x 16,384 18.4 / 17.4; 1536
  // bytes x 64 13.5 / 12.6, x 4,096 17.2 / 16.6; 4112 bytes x 1 12.6 / 11.6, x 1,024 20.3 / 19.7; 8 KB x 8 15.5 / 15.8, x 1,024 26.7 / 25.6; 32 KB
  // x 2 25.4 / 27.0, x 8 33.3 / 34.9, x 64 45.7 / 45.5, x 4,096 78.4 / 75.7; a flat table: 1040 bytes x 4,032 15.0 / 14.5, x 16,384 19.2 / 18.9;
  // 4112 bytes x 1,024 19.8 / 18.9, x 4,096 22.3 / 21.3; 8 KB x 4,096 30.1 / 27.6; 32 KB x 8 32.7 / 34.3.  Zipf 1.05 sooner everywhere but
  // for one row of 32 KB, by up to 14 %.
  const size_t out_bytes = n * row_bytes;
  DoneWords done = nt && !flat ? DoneWords{} : request.take(grid, Telling::kSooner, n);
  UGK_REQUIRE(!request.counted(), "ugk_extract_mix: a launch that leaves no words cannot take its count from the device");
  if (!done.tag) done.words = reinterpret_cast<unsigned long long *>(counts);
  if (num_groups) *num_groups = done.tag ? 0 : grid;
  const ugk_stage_t no_stage{};
  const bool few = KIND == 1 ? n <= 4096 : likely <= slots * 8;
  const bool keep = row_bytes <= 64 || out_bytes <= (size_t)64 << 20;
#define UGK_GO4(L, W, R, NT, KEEP, ST)                                                                              \
  hipLaunchKernelGGL((extract_mix_kernel<K, KIND, L, W, R, NT, KEEP, ST>), dim3(grid), dim3(kBlock), 0, st, t, keys, n,     \
                     cache, cache_rows, host, host_rows, out, f_row, status, host_mirror, Ending<NT>(done),        \
                     ST ? *stage : no_stage)
#define UGK_GO3(L, W, R, NT, KEEP)               \
  do {                                           \
    if (stage) UGK_GO4(L, W, R, NT, KEEP, true); \
    else UGK_GO4(L, W, R, NT, KEEP, false);      \
  } while (0)
#define UGK_ROWS(L, W, R)                                \
  do {                                                   \
    if constexpr (L > 4) {                               \
      if (done.tag && !keep) {                           \
        UGK_GO3(L, W, R, kThrough, false);               \
        break;                                           \
      }                                                  \
    }                                                    \
    if (done.tag) UGK_GO3(L, W, R, kThrough, true);      \
    else if (nt) UGK_GO3(L, W, R, kStreaming, false);    \
    else UGK_GO3(L, W, R, kOrdinary, false);             \
  } while (0)
#define UGK_GO2(L, W)                                             \
  do {                                                            \
    if constexpr (mix_rows(L, W) == 8 && (KIND == 1 || W == 16)) { \
      if (!few) {                                                 \
        UGK_ROWS(L, W, 4);                                        \
        break;                                                    \
      }                                                           \
    }                                                             \
    UGK_ROWS(L, W, mix_rows(L, W));                               \
  } while (0)
#define UGK_FLAT(W)                                                \
  do {                                                             \
    if (done.tag && keep) UGK_GO4(0, W, 4, kThrough, true, false); \
    else if (done.tag) UGK_GO4(0, W, 4, kThrough, false, false);   \
    else UGK_GO4(0, W, 4, kOrdinary, false, false);                \
  } while (0)
#define UGK_GO(L)                                   \
  do {                                              \
    if constexpr (kWave / L <= 8) {                 \
      if (kpw == 8) {                               \
        UGK_GO2(L, 8);                              \
        break;                                      \
      }                                             \
    }                                               \
    if constexpr (kWave / L <= 16) {                \
      if (kpw == 16) {                              \
        UGK_GO2(L, 16);                             \
        break;                                      \
      }                                             \
    }                                               \
    if constexpr (kWave / L <= 32) {                \
      if (kpw == 32) {                              \
        UGK_GO2(L, 32);                             \
        break;                                      \
      }                                             \
    }                                               \
    UGK_GO2(L, kWave);                              \
  } while (0)
  if (flat) {  // ordinary stores whatever the size (see flat_copy)
    if (kpw == 8) UGK_FLAT(8);
    else if (kpw == 16) UGK_FLAT(16);
    else if (kpw == 32) UGK_FLAT(32);
    else UGK_FLAT(kWave);
  } else if (vpr <= 1) UGK_GO2(1, kWave);
  else if (vpr <= 2) UGK_GO(2);
  else if (vpr <= 4) UGK_GO(4);
  else if (vpr <= 8) UGK_GO(8);
  else if (vpr <= 16) UGK_GO(16);
  else if (vpr <= 32) UGK_GO(32);
  else UGK_GO(64);
#undef UGK_GO
#undef UGK_GO2
#undef UGK_ROWS
#undef UGK_GO3
#undef UGK_GO4
#undef UGK_FLAT
  UGK_HIP(hipGetLastError());
  return 0;
}

template <typename K>
int extract_mix(ugk_table_t t, const K *keys, size_t n, const void *cache, uint64_t cache_rows, const void *host,
                uint64_t host_rows, void *out, size_t row_bytes, uint32_t *status, uint32_t *host_mirror,
                uint64_t *counts, uint32_t *num_groups, uint32_t others_hint, const ugk_stage_t *stage, void *stream) {
  DoneRequest request;
  if (num_groups) *num_groups = 0;
  if (n == 0) return 0;
  UGK_REQUIRE(keys && out && status, "ugk_extract_mix: null keys, output or status");
  UGK_REQUIRE((uintptr_t)counts % 8 == 0, "ugk_extract_mix: the count words must be 8-byte aligned");
  UGK_REQUIRE(n <= 0xffffffffull, "ugk_extract_mix: batch of %zu keys exceeds 2^32", n);
  UGK_REQUIRE(t.kind >= 1 && t.kind <= 3, "ugk_extract_mix: table kind %d is not flat(1), hash(2) or compact hash(3)", t.kind);
  UGK_REQUIRE(t.table && t.size, "ugk_extract_mix: empty table");
  if (t.kind >= 2)
    UGK_REQUIRE(t.size % (t.kind == 2 ? 8 : 16) == 0 && (uintptr_t)t.table % 128 == 0,
                "ugk_extract_mix: hash table must be 128-byte aligned with whole 128-byte lines of buckets");
  UGK_REQUIRE(cache_rows == 0 || cache, "ugk_extract_mix: null cache with %llu rows", (unsigned long long)cache_rows);
  UGK_REQUIRE(host_rows == 0 || host, "ugk_extract_mix: null host table with %llu rows",
              (unsigned long long)host_rows);
  const uintptr_t align = (uintptr_t)cache | (uintptr_t)host | (uintptr_t)out | (uintptr_t)row_bytes;
  const bool flat = align % 16 != 0;
  UGK_REQUIRE(row_bytes > 0 && (!flat || row_bytes <= kFlatMaxBytes), "ugk_extract_mix: row_bytes %zu out of range",
              row_bytes);
  UGK_REQUIRE(!flat || (flat_row_ok(align, row_bytes) && !stage),
              "ugk_extract_mix: rows and buffers must be multiples of 16 bytes, or without a stage of 4 bytes with rows "
              "of at least %u (row_bytes=%zu)",
              kFlatMinBytes, row_bytes);
  if (stage) {
    UGK_REQUIRE(stage->rows_dev && stage->owner_dev, "ugk_extract_mix_staged: null stage");
    UGK_REQUIRE(((stage->mask + 1) & stage->mask) == 0, "ugk_extract_mix_staged: the stage needs a power of two of entries");
    UGK_REQUIRE(stage->epoch != 0, "ugk_extract_mix_staged: the launch tag must be non-zero");
    UGK_REQUIRE((uintptr_t)stage->rows_dev % 16 == 0 && (uintptr_t)stage->owner_dev % 8 == 0,
                "ugk_extract_mix_staged: misaligned stage");
  }
  if (t.kind == 1)
    return extract_mix_lpr<K, 1>(t, keys, n, cache, cache_rows, host, host_rows, out, row_bytes, flat, status,
                                 host_mirror, counts, num_groups, others_hint, stage, request, as_stream(stream));
  if (t.kind == 2)
    return extract_mix_lpr<K, 2>(t, keys, n, cache, cache_rows, host, host_rows, out, row_bytes, flat, status,
                                 host_mirror, counts, num_groups, others_hint, stage, request, as_stream(stream));
  return extract_mix_lpr<K, 3>(t, keys, n, cache, cache_rows, host, host_rows, out, row_bytes, flat, status,
                               host_mirror, counts, num_groups, others_hint, stage, request, as_stream(stream));
}

// The workspace is laid out by its own size, not by the batch's: `cap` slot words, then cap / 2 words of unique ids by
// first occurrence (a batch may bring at most cap / 2 keys).  Batches of any size that share a workspace therefore agree
// on what is a slot and what is not, which the epoch tags rely on.
size_t dedup_capacity_of_workspace(size_t bytes) {
  size_t cap = 0;
  for (size_t c = 1024; c * 10 + 64 <= bytes; c <<= 1) cap = c;
  return cap;
}

template <typename K>
int dedup(const K *keys, size_t n, void *workspace, size_t workspace_bytes, uint32_t epoch, const uint32_t *epoch_dev,
          K *unique_out, uint32_t *inverse, uint32_t *rep_of, uint32_t *n_unique, uint32_t *n_unique_host,
          uint32_t *next_n_unique, void *stream) {
  if (n == 0) return 0;
  UGK_REQUIRE(keys && workspace && unique_out && inverse && n_unique, "ugk_dedup: null pointer");
  UGK_REQUIRE(epoch != 0 || epoch_dev, "ugk_dedup: epoch must be non-zero");
  UGK_REQUIRE(n <= 0x7fffffffull, "ugk_dedup: batch of %zu keys exceeds 2^31", n);
  UGK_REQUIRE((uintptr_t)workspace % 8 == 0, "ugk_dedup: workspace must be 8-byte aligned");
  const size_t cap = dedup_capacity_of_workspace(workspace_bytes);
  UGK_REQUIRE(cap >= 2 * n, "ugk_dedup: a workspace of %zu bytes holds batches of up to %zu keys, this one has %zu",
              workspace_bytes, cap / 2, n);
  if (n <= kSmallBatch) {
#define UGK_GO(ITEMS)                                                                                                          \
  hipLaunchKernelGGL((dedup_small_kernel<K, ITEMS>), dim3(1), dim3(kSmallBlock), 0, as_stream(stream), keys, (uint32_t)n, unique_out, \
                     inverse, rep_of, n_unique, n_unique_host, next_n_unique)
    if (n <= kSmallBlock) UGK_GO(1);
    else if (n <= 2 * kSmallBlock) UGK_GO(2);
    else UGK_GO(4);
#undef UGK_GO
    UGK_HIP(hipGetLastError());
    return 0;
  }
  unsigned long long *slots = reinterpret_cast<unsigned long long *>(workspace);
  uint32_t *uid_of = reinterpret_cast<uint32_t *>(slots + cap);
  // 256-key tiles while larger ones would leave compute units idle, 512-key ones up to twice as many keys; beyond that the
  // larger tile wins, because more of a skewed batch's duplicates meet in LDS.  us with the set cleared in front of it (about
  // 5 of them), 256 / 512 / 1024-key tiles: 65,536 keys uniform 29 / 38 / 57, Zipf 0.9 27 / 30 / 41, Zipf 1.3 18 / 18 / 20;
  // 100,000 keys 27 / 32 / 46, 29 / 28 / 36, 24 / 21 / 21; 200,000 keys 36 / 38 / 51, 43 / 35 / 39, 39 / 29 / 23.
  const size_t per_cu = (size_t)cu_count() * kBlock;
  const int items = n <= per_cu ? 1 : n <= 2 * per_cu ? 2 : kItems;
  const size_t tile = (size_t)kBlock * items;
  const unsigned claim_grid = clamp_grid((n + tile - 1) / tile, 0);
  if (items == 1)
    hipLaunchKernelGGL((dedup_claim_kernel<K, 1>), dim3(claim_grid), dim3(kBlock), 0, as_stream(stream), keys, n,
                       slots, cap - 1, epoch, epoch_dev, uid_of, unique_out, inverse, rep_of, n_unique);
  else if (items == 2)
    hipLaunchKernelGGL((dedup_claim_kernel<K, 2>), dim3(claim_grid), dim3(kBlock), 0, as_stream(stream), keys, n,
                       slots, cap - 1, epoch, epoch_dev, uid_of, unique_out, inverse, rep_of, n_unique);
  else
    hipLaunchKernelGGL((dedup_claim_kernel<K, kItems>), dim3(claim_grid), dim3(kBlock), 0, as_stream(stream), keys, n,
                       slots, cap - 1, epoch, epoch_dev, uid_of, unique_out, inverse, rep_of, n_unique);
  UGK_HIP(hipGetLastError());
  const unsigned grid = clamp_grid((n + kBlock - 1) / kBlock, 0);
  hipLaunchKernelGGL(dedup_resolve_kernel, dim3(grid), dim3(kBlock), 0, as_stream(stream), n, uid_of, inverse,
                     n_unique, n_unique_host, next_n_unique);
  UGK_HIP(hipGetLastError());
  return 0;
}

}  // namespace
// an empty launch: what it costs is the load of this file's code object onto the device (see ugk_preload_kernels)
namespace {
__global__ void preload_partition_kernel() {}
}  // namespace
void preload_partition(hipStream_t stream) { hipLaunchKernelGGL(preload_partition_kernel, dim3(1), dim3(1), 0, stream); }
}  // namespace ugk

using namespace ugk;

extern "C" {

int ugk_classify_u32(ugk_table_t t, const uint32_t *keys_dev, size_t n, uint64_t host_rows, const uint32_t *dst_map_dev,
                     ugk_idx_t *idx_dev, uint32_t *counts_dev, uint32_t *next_counts_dev, uint32_t *status_dev,
                     uint32_t *host_mirror, void *stream) {
  return classify<uint32_t>(t, keys_dev, n, host_rows, dst_map_dev, idx_dev, counts_dev, next_counts_dev, status_dev,
                            host_mirror, stream);
}
int ugk_classify_i64(ugk_table_t t, const int64_t *keys_dev, size_t n, uint64_t host_rows, const uint32_t *dst_map_dev,
                     ugk_idx_t *idx_dev, uint32_t *counts_dev, uint32_t *next_counts_dev, uint32_t *status_dev,
                     uint32_t *host_mirror, void *stream) {
  return classify<int64_t>(t, keys_dev, n, host_rows, dst_map_dev, idx_dev, counts_dev, next_counts_dev, status_dev,
                           host_mirror, stream);
}

int ugk_nonlocal_flags_u32(ugk_table_t t, const uint32_t *keys_dev, size_t n, uint64_t *flags_dev, void *stream) {
  return nonlocal_flags<uint32_t>(t, keys_dev, n, flags_dev, stream);
}
int ugk_nonlocal_flags_i64(ugk_table_t t, const int64_t *keys_dev, size_t n, uint64_t *flags_dev, void *stream) {
  return nonlocal_flags<int64_t>(t, keys_dev, n, flags_dev, stream);
}
int ugk_select_keys_u32(const uint32_t *keys_dev, const uint32_t *sel_dev, size_t m, uint32_t *out_dev, void *stream) {
  return select_keys<uint32_t>(keys_dev, sel_dev, m, out_dev, stream);
}
int ugk_select_keys_i64(const int64_t *keys_dev, const uint32_t *sel_dev, size_t m, int64_t *out_dev, void *stream) {
  return select_keys<int64_t>(keys_dev, sel_dev, m, out_dev, stream);
}

unsigned ugk_extract_mix_max_groups(void) { return clamp_grid(~(size_t)0, 0); }

int ugk_extract_mix_u32(ugk_table_t t, const uint32_t *keys_dev, size_t n, const void *cache_dev, uint64_t cache_rows,
                        const void *host_dev, uint64_t host_rows, void *out_dev, size_t row_bytes,
                        uint32_t *status_dev, uint32_t *host_mirror, uint64_t *group_counts_host,
                        uint32_t *num_groups_host, uint32_t others_hint, void *stream) {
  return extract_mix<uint32_t>(t, keys_dev, n, cache_dev, cache_rows, host_dev, host_rows, out_dev, row_bytes,
                               status_dev, host_mirror, group_counts_host, num_groups_host, others_hint, nullptr,
                               stream);
}
int ugk_extract_mix_i64(ugk_table_t t, const int64_t *keys_dev, size_t n, const void *cache_dev, uint64_t cache_rows,
                        const void *host_dev, uint64_t host_rows, void *out_dev, size_t row_bytes,
                        uint32_t *status_dev, uint32_t *host_mirror, uint64_t *group_counts_host,
                        uint32_t *num_groups_host, uint32_t others_hint, void *stream) {
  return extract_mix<int64_t>(t, keys_dev, n, cache_dev, cache_rows, host_dev, host_rows, out_dev, row_bytes,
                              status_dev, host_mirror, group_counts_host, num_groups_host, others_hint, nullptr,
                              stream);
}
int ugk_extract_mix_staged_u32(ugk_table_t t, const uint32_t *keys_dev, size_t n, const void *cache_dev,
                               uint64_t cache_rows, const void *host_dev, uint64_t host_rows, void *out_dev,
                               size_t row_bytes, uint32_t *status_dev, uint32_t *host_mirror,
                               uint64_t *group_counts_host, uint32_t *num_groups_host, uint32_t others_hint,
                               ugk_stage_t stage, void *stream) {
  return extract_mix<uint32_t>(t, keys_dev, n, cache_dev, cache_rows, host_dev, host_rows, out_dev, row_bytes,
                               status_dev, host_mirror, group_counts_host, num_groups_host, others_hint, &stage,
                               stream);
}
int ugk_extract_mix_staged_i64(ugk_table_t t, const int64_t *keys_dev, size_t n, const void *cache_dev,
                               uint64_t cache_rows, const void *host_dev, uint64_t host_rows, void *out_dev,
                               size_t row_bytes, uint32_t *status_dev, uint32_t *host_mirror,
                               uint64_t *group_counts_host, uint32_t *num_groups_host, uint32_t others_hint,
                               ugk_stage_t stage, void *stream) {
  return extract_mix<int64_t>(t, keys_dev, n, cache_dev, cache_rows, host_dev, host_rows, out_dev, row_bytes,
                              status_dev, host_mirror, group_counts_host, num_groups_host, others_hint, &stage,
                              stream);
}

size_t ugk_dedup_workspace_bytes(size_t n) { return dedup_capacity(n) * 10 + 64; }

int ugk_dedup_static(const void *keys_dev, uint32_t key_bytes, size_t n, void *unique_out_dev,
                     uint32_t *inverse_out_dev, uint32_t *rep_out_dev, uint32_t *n_unique_dev, uint32_t *n_unique_host,
                     void *stream) {
  UGK_REQUIRE(key_bytes == 4 || key_bytes == 8, "ugk_dedup_static: keys of %u bytes (4 or 8 are supported)", key_bytes);
  UGK_REQUIRE(n_unique_dev, "ugk_dedup_static: null count word");
  UGK_REQUIRE(n <= UGK_DEDUP_STATIC_MAX_KEYS,
              "ugk_dedup_static: a batch of %zu keys exceeds the %zu the static scratch is sized for "
              "(use ugk_dedup_u32 / ugk_dedup_i64 with a workspace of your own)",
              n, (size_t)UGK_DEDUP_STATIC_MAX_KEYS);
  // the device address of this GPU's copy of the array, looked up once per device with that device current
  static std::mutex mu;
  static unsigned char *base_of[64] = {nullptr};
  int dev = 0;
  UGK_HIP(hipGetDevice(&dev));
  UGK_REQUIRE(dev >= 0 && dev < 64, "ugk_dedup_static: device %d out of range", dev);
  unsigned char *base = nullptr;
  {
    std::lock_guard<std::mutex> guard(mu);
    if (base_of[dev] == nullptr) {
      void *p = nullptr;
      UGK_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
      UGK_REQUIRE(p != nullptr, "ugk_dedup_static: no device address for the static scratch");
      base_of[dev] = static_cast<unsigned char *>(p);
    }
    base = base_of[dev];
  }
  uint32_t *epoch_dev = reinterpret_cast<uint32_t *>(base);
  unsigned char *ws = base + UGK_DEDUP_STATIC_HEADER;
  const size_t cap = dedup_capacity_of_workspace(UGK_DEDUP_STATIC_WS_BYTES);
  hipLaunchKernelGGL(static_wrap_kernel, dim3(clamp_grid(1024, 0)), dim3(kBlock), 0, as_stream(stream),
                     epoch_dev, reinterpret_cast<unsigned long long *>(ws), cap);
  UGK_HIP(hipGetLastError());
  hipLaunchKernelGGL(static_epoch_kernel, dim3(1), dim3(1), 0, as_stream(stream), epoch_dev, n_unique_dev,
                     n_unique_host);
  UGK_HIP(hipGetLastError());
  if (n == 0) return 0;
  if (key_bytes == 4)
    return dedup<uint32_t>(static_cast<const uint32_t *>(keys_dev), n, ws, UGK_DEDUP_STATIC_WS_BYTES, 0, epoch_dev,
                           static_cast<uint32_t *>(unique_out_dev), inverse_out_dev, rep_out_dev, n_unique_dev,
                           n_unique_host, nullptr, stream);
  return dedup<int64_t>(static_cast<const int64_t *>(keys_dev), n, ws, UGK_DEDUP_STATIC_WS_BYTES, 0, epoch_dev,
                        static_cast<int64_t *>(unique_out_dev), inverse_out_dev, rep_out_dev, n_unique_dev,
                        n_unique_host, nullptr, stream);
}

int ugk_dedup_rotating(const void *keys_dev, uint32_t key_bytes, size_t n, void *workspace_dev, size_t workspace_bytes,
                       uint32_t epoch, void *unique_out_dev, uint32_t *inverse_out_dev, uint32_t *rep_out_dev,
                       uint32_t *n_unique_dev, uint32_t *next_n_unique_dev, uint32_t *n_unique_host, void *stream) {
  UGK_REQUIRE(key_bytes == 4 || key_bytes == 8, "ugk_dedup_rotating: keys of %u bytes (4 or 8 are supported)", key_bytes);
  UGK_REQUIRE(next_n_unique_dev && next_n_unique_dev != n_unique_dev, "ugk_dedup_rotating: one count word for two calls");
  if (key_bytes == 4)
    return dedup<uint32_t>(static_cast<const uint32_t *>(keys_dev), n, workspace_dev, workspace_bytes, epoch, nullptr,
                           static_cast<uint32_t *>(unique_out_dev), inverse_out_dev, rep_out_dev, n_unique_dev,
                           n_unique_host, next_n_unique_dev, stream);
  return dedup<int64_t>(static_cast<const int64_t *>(keys_dev), n, workspace_dev, workspace_bytes, epoch, nullptr,
                        static_cast<int64_t *>(unique_out_dev), inverse_out_dev, rep_out_dev, n_unique_dev, n_unique_host,
                        next_n_unique_dev, stream);
}

int ugk_dedup_u32(const uint32_t *keys_dev, size_t n, void *workspace_dev, size_t workspace_bytes, uint32_t epoch,
                  uint32_t *unique_out_dev, uint32_t *inverse_out_dev, uint32_t *rep_out_dev, uint32_t *n_unique_dev,
                  uint32_t *n_unique_host, void *stream) {
  return dedup<uint32_t>(keys_dev, n, workspace_dev, workspace_bytes, epoch, nullptr, unique_out_dev, inverse_out_dev,
                         rep_out_dev, n_unique_dev, n_unique_host, nullptr, stream);
}
int ugk_dedup_i64(const int64_t *keys_dev, size_t n, void *workspace_dev, size_t workspace_bytes, uint32_t epoch,
                  int64_t *unique_out_dev, uint32_t *inverse_out_dev, uint32_t *rep_out_dev, uint32_t *n_unique_dev,
                  uint32_t *n_unique_host, void *stream) {
  return dedup<int64_t>(keys_dev, n, workspace_dev, workspace_bytes, epoch, nullptr, unique_out_dev, inverse_out_dev,
                        rep_out_dev, n_unique_dev, n_unique_host, nullptr, stream);
}

}  // extern "C"
