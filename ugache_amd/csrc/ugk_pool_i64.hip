// Pooled extraction of 8-byte ids (ugk_pool.cuh).
#include "ugk_pool.cuh"

namespace ugk {
// an empty launch: what it costs is the load of this file's code object onto the device (see ugk_preload_kernels)
namespace {
__global__ void preload_pool_i64_kernel() {}
}  // namespace
void preload_pool_i64(hipStream_t stream) { hipLaunchKernelGGL(preload_pool_i64_kernel, dim3(1), dim3(1), 0, stream); }
}  // namespace ugk

using namespace ugk;

extern "C" {

int ugk_extract_pool_i64(ugk_table_t t, const int64_t *ids_dev, const int64_t *seg_off_dev, const float *weights_dev,
                         size_t n_rows, uint64_t nnz, int combiner, int elem_bytes, const void *cache_dev,
                         uint64_t cache_rows, const void *host_dev, uint64_t host_rows, void *out_dev, size_t row_bytes,
                         uint32_t *status_dev, uint32_t *host_mirror, uint64_t *group_counts_host,
                         uint32_t *num_groups_host, void *stream) {
  return extract_pool<int64_t>(t, ids_dev, seg_off_dev, weights_dev, n_rows, nnz, combiner, elem_bytes, cache_dev,
                               cache_rows, host_dev, host_rows, out_dev, row_bytes, 0.f, status_dev, host_mirror,
                               group_counts_host, num_groups_host, stream);
}

int ugk_extract_pool_clip_i64(ugk_table_t t, const int64_t *ids_dev, const int64_t *seg_off_dev,
                              const float *weights_dev, size_t n_rows, uint64_t nnz, int combiner, int elem_bytes,
                              float max_norm, const void *cache_dev, uint64_t cache_rows, const void *host_dev,
                              uint64_t host_rows, void *out_dev, size_t row_bytes, uint32_t *status_dev,
                              uint32_t *host_mirror, uint64_t *group_counts_host, uint32_t *num_groups_host,
                              void *stream) {
  return extract_pool<int64_t>(t, ids_dev, seg_off_dev, weights_dev, n_rows, nnz, combiner, elem_bytes, cache_dev,
                               cache_rows, host_dev, host_rows, out_dev, row_bytes, max_norm, status_dev, host_mirror,
                               group_counts_host, num_groups_host, stream);
}

}  // extern "C"
