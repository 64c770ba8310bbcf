// What gemm.hip and gemm_list.hip ask of the small-tile kernel (gemm_deep.hip).
#pragma once
#include "common.h"

namespace mi {

constexpr int DEEP_MAX = 8;
struct DeepProblem {
    const int8_t *qx, *qw;
    const float *sx, *sw;
    void *out;
    int M, N, K;
    // filled in by the launch: first workgroup, tiles, row tiles and what divides by their number
    int first, tiles, tiles_m;
    unsigned magic;
};

// microseconds that the launch would take; *which is the tile to pass on
float deep_estimate(int M, int N, int K, int cus, int *which);
int deep_fine(int M, int N, int K, int cus, int coarse, float tiled_us);   // the tile after all, or -1: not this kernel
void deep_tile(int which, int32_t *rows, int32_t *cols);
bool deep_fits(int which, int M, int N);   // no more tiles than the kernel's arithmetic covers
float deep_batch_estimate(const int64_t *mnk, const int *idx, int n, int cus, int *which);   // problems idx[0 .. n-1], longest K first

template <bool DEQ>
int32_t launch_deep(int which, const int8_t *qx, const float *sx, const int8_t *qw, const float *sw, int32_t *acc, float *y,
                    int64_t M, int64_t N, int64_t K, hipStream_t s);
template <bool DEQ>
int32_t launch_deep_batch(int which, const DeepProblem *p, int n, hipStream_t s);

}  // namespace mi
