// The merge of the partial results that the attention kernels leave, for the merge kernels (attention.hip) and for the projection of
// one token that merges them itself (gemv.hip): the same operations in the same order, so the same bits.
#pragma once
#include "common.h"

namespace mi {
namespace attn {

constexpr int MERGE_D = 128;

// The splits of one lane's eight elements, requested with load and added with add.  ALL: MOST of them; otherwise at most, and the last
// one is read in place of those that are not there
template <int MOST, bool ALL>
struct Partials {
    float ms[MOST], ls[MOST];
    float4 lo[MOST], hi[MOST];

    __device__ __forceinline__ void load(const float *__restrict__ ml0, const float *__restrict__ po0, int splits, int hl, int j)
    {
#pragma unroll
        for (int i = 0; i < MOST; ++i) {
            const int s = ALL ? i : min(i, splits - 1);
            ms[i] = ml0[s * 8 + hl];
            ls[i] = ml0[s * 8 + 4 + hl];
            lo[i] = *reinterpret_cast<const float4 *>(po0 + s * 4 * MERGE_D + 4 * j);
            hi[i] = *reinterpret_cast<const float4 *>(po0 + s * 4 * MERGE_D + 64 + 4 * j);
        }
    }
    __device__ __forceinline__ void add(int splits, float (&v)[8], float &l) const
    {
        float mx = ms[0];
#pragma unroll
        for (int s = 1; s < MOST; ++s) mx = fmaxf(mx, ms[s]);
#pragma unroll
        for (int s = 0; s < MOST; ++s) {
            const float w = ((!ALL && s >= splits) || ms[s] == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(ms[s] - mx);   // empty split
            l = __builtin_fmaf(ls[s], w, l);
            v[0] = __builtin_fmaf(lo[s].x, w, v[0]); v[1] = __builtin_fmaf(lo[s].y, w, v[1]);
            v[2] = __builtin_fmaf(lo[s].z, w, v[2]); v[3] = __builtin_fmaf(lo[s].w, w, v[3]);
            v[4] = __builtin_fmaf(hi[s].x, w, v[4]); v[5] = __builtin_fmaf(hi[s].y, w, v[5]);
            v[6] = __builtin_fmaf(hi[s].z, w, v[6]); v[7] = __builtin_fmaf(hi[s].w, w, v[7]);
        }
    }
};

// the sums brought to weight 1
__device__ __forceinline__ void normalize_row(float l, float (&v)[8])
{
    const float rl = l > 0.0f ? 1.0f / l : 0.0f;   // a sequence of length 0 gives a row of zeros
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] *= rl;
}

// Merge of the splits of one (b, h) row by the 16 lanes that own it (lane j: elements 4j..4j+3 and 64+4j..).
// SP > 0: the split count is known at compile time and every load of the row goes out before the first use (one
// memory round trip); SP < 0: the same for a count of at most -SP (the last split is read in place of those that are not there).
// Returns the normalized row in the rotated basis of V.
template <int SP, int BATCH = 8>
__device__ __forceinline__ void merge_row(const float *__restrict__ part_o, const float *__restrict__ part_ml,
                                          int splits_rt, int64_t bkv, int hl, int j, float (&v)[8])
{
    constexpr int MOST = SP < 0 ? -SP : SP;
    const int splits = SP > 0 ? SP : splits_rt;
    const float *ml0 = part_ml + bkv * splits * 8;
    const float *po0 = part_o + (bkv * splits * 4 + hl) * MERGE_D;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = 0.0f;
    float l = 0.0f;
    if constexpr (MOST > 0) {
        Partials<MOST, (SP > 0)> part;
        part.load(ml0, po0, splits, hl, j);
        // all of them before the first use: the compiler otherwise saves registers and makes two round trips of it.  us of attention
        // and merge, one sequence in spans of 256 tokens, 10 splits 10.4 -> 8.2, 14 10.5 -> 8.6, 16 8.9 -> 8.1.  (Not in workgroups
        // of up to 1024 threads, which have 128 registers.)
        if constexpr (BATCH == 16) __builtin_amdgcn_sched_barrier(0);
        part.add(splits, v, l);
    } else {
        // any split count: the maxima first (one round trip), then the partials in batches of BATCH whose loads all
        // go out before the first use
        float mx = -INFINITY;
        for (int s0 = 0; s0 < splits; s0 += BATCH) {
            float ms[BATCH];
#pragma unroll
            for (int i = 0; i < BATCH; ++i) ms[i] = ml0[min(s0 + i, splits - 1) * 8 + hl];
#pragma unroll
            for (int i = 0; i < BATCH; ++i) mx = fmaxf(mx, ms[i]);
        }
        for (int s0 = 0; s0 < splits; s0 += BATCH) {
            float ms[BATCH], ls[BATCH];
            float4 lo[BATCH], hi[BATCH];
#pragma unroll
            for (int i = 0; i < BATCH; ++i) {
                const int s = min(s0 + i, splits - 1);
                ms[i] = ml0[s * 8 + hl];
                ls[i] = ml0[s * 8 + 4 + hl];
                lo[i] = *reinterpret_cast<const float4 *>(po0 + s * 4 * MERGE_D + 4 * j);
                hi[i] = *reinterpret_cast<const float4 *>(po0 + s * 4 * MERGE_D + 64 + 4 * j);
            }
#pragma unroll
            for (int i = 0; i < BATCH; ++i) {
                const float w = (s0 + i >= splits || ms[i] == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(ms[i] - mx);
                l = __builtin_fmaf(ls[i], w, l);
                v[0] = __builtin_fmaf(lo[i].x, w, v[0]); v[1] = __builtin_fmaf(lo[i].y, w, v[1]);
                v[2] = __builtin_fmaf(lo[i].z, w, v[2]); v[3] = __builtin_fmaf(lo[i].w, w, v[3]);
                v[4] = __builtin_fmaf(hi[i].x, w, v[4]); v[5] = __builtin_fmaf(hi[i].y, w, v[5]);
                v[6] = __builtin_fmaf(hi[i].z, w, v[6]); v[7] = __builtin_fmaf(hi[i].w, w, v[7]);
            }
        }
    }
    normalize_row(l, v);
}

}  // namespace attn
}  // namespace mi
