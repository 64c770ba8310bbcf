// What gemm_list.hip asks of the kernel that walks a list of 256 x 128 tiles (gemm_stream.hip).
#pragma once
#include "common.h"

namespace mi {

typedef int v2i __attribute__((ext_vector_type(2)));

constexpr int STREAM_MAX = 8;
constexpr int STREAM_BN = 128;   // columns of a tile; it has 256 rows
// The shortest K that a list may hold.  The kernel's two areas of scales need more stages of 128 bytes a tile than it has stage
// buffers, three: four or more, K >= 512.  1024 is the line that the rule of gemm_list.hip was measured with.
constexpr int64_t STREAM_MIN_K = 1024;
struct StreamProblem {
    const int8_t *qx, *qw;
    const float *sx, *sw;
    void *out;
    int M, N, K, pad;
};
struct StreamBatch {
    StreamProblem p[STREAM_MAX];
};

template <bool DEQ>
int32_t launch_stream(const StreamBatch &b, const v2i *lists, int grid, int per_wg, hipStream_t s);

}  // namespace mi
