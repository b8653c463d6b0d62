// Pooled extraction of 4-byte ids (ugk_pool.cuh) and the offsets of a pooled lookup (ugk_segment_offsets_i64).
#include "ugk_pool.cuh"

namespace ugk {
namespace {

// seg_off[r] = the number of entries whose row is below r: lane i owns the offsets of the rows that begin between
// entry i - 1 and entry i.  That is one offset where every row has an entry, which the lane writes itself; a run of
// rows without entries is written by the whole wavefront, 64 offsets a step.
__global__ __launch_bounds__(kBlock) void segment_offsets_kernel(const long long *__restrict__ rows, size_t nnz,
                                                                 size_t n_rows, long long *__restrict__ seg_off,
                                                                 uint32_t *status, uint32_t *host_mirror) {
  const size_t stride = (size_t)gridDim.x * kBlock;
  const int lane = (int)lane_id();
  for (size_t base = (size_t)blockIdx.x * kBlock + threadIdx.x - lane; base <= nnz; base += stride) {  // wavefront-uniform
    const size_t i = base + lane;
    long long prev = 0, cur = -1;  // an empty run for the lanes past the end
    if (i <= nnz) {
      prev = i == 0 ? -1 : rows[i - 1];
      cur = i == nnz ? (long long)n_rows : rows[i];
      // entries out of order or outside [0, n_rows): flagged; what is written stays inside seg_off
      if (cur < prev || cur < 0 || (i > 0 && prev < 0) || (i < nnz && cur >= (long long)n_rows) ||
          prev >= (long long)n_rows) {
        if (status) atomicOr(status, UGK_ST_BAD_SEGMENT);
        if (host_mirror) tell_host<uint32_t>(host_mirror, UGK_ST_BAD_SEGMENT);
        prev = 0, cur = -1;
      }
    }
    const long long first = prev + 1, count = cur - prev;  // rows first .. first + count - 1 begin at entry i
    if (count == 1) seg_off[first] = (long long)i;
    for (unsigned long long runs = __ballot(count > 1); runs != 0ull; runs &= runs - 1ull) {
      const int src = __ffsll((long long)runs) - 1;
      const long long f = (long long)shfl64((uint64_t)first, src), c = (long long)shfl64((uint64_t)count, src);
      const long long at = (long long)(base + src);
      for (long long r = lane; r < c; r += kWave) seg_off[f + r] = at;
    }
  }
}

}  // namespace
// an empty launch: what it costs is the load of this file's code object onto the device (see ugk_preload_kernels)
namespace {
__global__ void preload_pool_kernel() {}
}  // namespace
void preload_pool(hipStream_t stream) { hipLaunchKernelGGL(preload_pool_kernel, dim3(1), dim3(1), 0, stream); }
}  // namespace ugk

using namespace ugk;

extern "C" {

int ugk_segment_offsets_i64(const int64_t *sorted_rows_dev, size_t nnz, size_t n_rows, int64_t *seg_off_dev,
                            uint32_t *status_dev, uint32_t *host_mirror, void *stream) {
  UGK_REQUIRE(seg_off_dev, "ugk_segment_offsets: null output");
  UGK_REQUIRE(nnz == 0 || sorted_rows_dev, "ugk_segment_offsets: null rows");
  UGK_REQUIRE(nnz < ((uint64_t)1 << 62) && n_rows < ((uint64_t)1 << 62), "ugk_segment_offsets: sizes out of range");
  const unsigned grid = clamp_grid((nnz + 1 + kBlock - 1) / kBlock, 0);
  hipLaunchKernelGGL(segment_offsets_kernel, dim3(grid), dim3(kBlock), 0, as_stream(stream),
                     reinterpret_cast<const long long *>(sorted_rows_dev), nnz, n_rows,
                     reinterpret_cast<long long *>(seg_off_dev), status_dev, host_mirror);
  UGK_HIP(hipGetLastError());
  return 0;
}

int ugk_extract_pool_u32(ugk_table_t t, const uint32_t *ids_dev, const int64_t *seg_off_dev, const float *weights_dev,
                         size_t n_rows, uint64_t nnz, int combiner, int elem_bytes, const void *cache_dev,
                         uint64_t cache_rows, const void *host_dev, uint64_t host_rows, void *out_dev, size_t row_bytes,
                         uint32_t *status_dev, uint32_t *host_mirror, uint64_t *group_counts_host,
                         uint32_t *num_groups_host, void *stream) {
  return extract_pool<uint32_t>(t, ids_dev, seg_off_dev, weights_dev, n_rows, nnz, combiner, elem_bytes, cache_dev,
                                cache_rows, host_dev, host_rows, out_dev, row_bytes, 0.f, status_dev, host_mirror,
                                group_counts_host, num_groups_host, stream);
}

int ugk_extract_pool_clip_u32(ugk_table_t t, const uint32_t *ids_dev, const int64_t *seg_off_dev,
                              const float *weights_dev, size_t n_rows, uint64_t nnz, int combiner, int elem_bytes,
                              float max_norm, const void *cache_dev, uint64_t cache_rows, const void *host_dev,
                              uint64_t host_rows, void *out_dev, size_t row_bytes, uint32_t *status_dev,
                              uint32_t *host_mirror, uint64_t *group_counts_host, uint32_t *num_groups_host,
                              void *stream) {
  return extract_pool<uint32_t>(t, ids_dev, seg_off_dev, weights_dev, n_rows, nnz, combiner, elem_bytes, cache_dev,
                                cache_rows, host_dev, host_rows, out_dev, row_bytes, max_norm, status_dev, host_mirror,
                                group_counts_host, num_groups_host, stream);
}

}  // extern "C"
