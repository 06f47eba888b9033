// edge_sort.hpp -- edge_list_to_csr by partition and sort (edge_sort.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace tg {

struct EdgeSortStatus {
    unsigned long long bad;  // first invalid endpoint, 2 * edge + (0 src, 1 dst); ~0: none
    int32_t dst_bad;         // whether a destination is outside [0, n)
    int32_t longest;         // edges of the largest bucket
    int32_t n_long;          // buckets past the short sort
};

// Whether the build takes a graph of these sizes, and its workspace.
bool edge_sort_fits(int64_t n, int64_t e);
size_t edge_sort_ws(int64_t n, int64_t e);
// Counts the buckets and checks the endpoints (destinations count towards
// `bad` where check_dst); synchronises s.
EdgeSortStatus edge_sort_count(int64_t n, int64_t e, const int32_t* src, const int32_t* dst,
                               bool check_dst, void* work, size_t work_bytes, hipStream_t s);
// Whether edge_sort_finish can follow: valid endpoints, no oversize bucket.
bool edge_sort_ready(const EdgeSortStatus& h);
void edge_sort_finish(const EdgeSortStatus& h, int64_t n, int64_t e, const int32_t* src,
                      const int32_t* dst, int32_t* row_ptr, int32_t* col_ind, float* val,
                      void* work, size_t work_bytes, hipStream_t s);

}  // namespace tg
