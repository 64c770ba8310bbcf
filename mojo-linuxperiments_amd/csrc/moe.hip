// MoE layer (workload elements a9 router, a10 dispatch, a11 grouped expert FFN).
//
//   route    : logits = x . wr^T (fixed fp32 order), top-k on logits, softmax over picks
//   dispatch : stable grouping of the T*topk (token, slot) pairs by expert
//   ffn      : qx = quant(FWHT128(x))                       once per token
//              per expert segment: g,u = qx . wg^T, qx . wu^T   (int8 MFMA, exact)
//                                  h = silu(g) * u              (fp32)  -> sorted order
//              hq = quant(FWHT256(h))                           per pair
//              per expert segment: out[pair] = hq . wd^T        (int8 MFMA, exact)
//              y[token] = sum_slot w[token,slot] * out[pair]    (fixed order, no atomics)
//
// The expert GEMMs are weight-streaming bound (each expert sees ~32 rows): a
// workgroup takes row chunks of 16 gate + 16 up rows (or 128 down rows), streams
// them from HBM once through wave-private LDS rings, and holds the expert's
// tokens, up to 64 at a time, in registers as MFMA B fragments.  The chunks of all
// experts that have tokens are dealt evenly to two workgroups a compute unit.
//
// Bound: HBM on the int8 expert weights, E * 3 * H * I bytes per layer call.
#include "common.h"
#include "lds_ops.h"
#include "fwht_core.h"

namespace mi {
namespace moe {

constexpr int MAX_TOPK = 8;
static int64_t align_up(int64_t v, int64_t a) { return (v + a - 1) / a * a; }
// ceil(2^32 / topk), or 0 where that does not divide every pair's number, which is less than 2^24 (see dispatch_pairs)
static uint32_t topk_magic(int topk)
{
    return topk < 2 || topk > 256 ? 0u : (uint32_t)(((1ull << 32) + (uint64_t)topk - 1) / (uint64_t)topk);
}
constexpr int64_t DISPATCH_MAX_WORDS = 36864;  // 144 KB of the 160 KB LDS


// ---------------------------------------------------------------- a9 router
// Workgroup = E/16 waves, 4 tokens.  Wave eg owns experts 16*eg .. 16*eg+15 for
// the 4 tokens: 64 (token, expert) dot products.  Lane l accumulates, for every
// one of them, the terms k = 256*j + 4*l + c (j ascending, c = 0..3) with one
// FMA each; the 64 lanes' partial sums are then combined by the butterfly
// l ^ 32, 16, 8, 4, 2, 1.  Instead of six shuffles per dot product, the
// butterfly is run "transposed": in the round with offset `off` a lane hands
// the half of its dot products whose index bit differs from its own lane bit
// to its partner and keeps the other half, so each addition joins exactly the
// two operands the plain butterfly would join (float add is commutative) and
// 63 shuffles finish 64 dot products.  Lane l ends with pair l.
template <int OFF, int N, int NP>
__device__ __forceinline__ void fold(float (&p)[NP], int lane)
{
    const bool hi = (lane & OFF) != 0;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        if constexpr (OFF == 32) {   // the exchange is one instruction
            const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(p[i]), __float_as_uint(p[i + N]), false, false);
            p[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
        } else if constexpr (OFF == 16) {
            const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(p[i]), __float_as_uint(p[i + N]), false, false);
            p[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
        } else {
            const float keep = hi ? p[i + N] : p[i];
            const float send = hi ? p[i] : p[i + N];
            p[i] = keep + __int_as_float(xor_lane_i<OFF>(__float_as_int(send)));
        }
    }
}

// grid = (T/16, E/EW): a workgroup of 4 waves covers 16 tokens x EW experts, so the router weights are read
// T/16 times and the activations E/EW times in all (both from L2), and every compute unit gets work.
// CQ > 0: the kernel also rotates (block 128) and quantizes the token rows for the expert FFN, a wave per row with CQ
// chunks per lane (H = 512 * CQ at most), the arithmetic of the stand-alone quantizer: the 16 tokens of a group are
// dealt to the waves of the group's workgroups, so that the layer launches one kernel less.
// EW = 8: a wave owns 8 experts for its 4 tokens (32 dot products a lane, half the registers, twice the workgroups):
// two waves share a SIMD where EW = 16 leaves one alone with its memory round trips (cfg4: 17.2 -> 13.8 us; four
// experts a wave, or loads two rounds ahead in three register sets, measured the same 13.8).  The first butterfly
// round (offset 32) is then the plain one; lanes l and l ^ 32 end with the same pair.
// EW = 1: few tokens.  Sixteen tokens are 16 workgroups at EW = 8, each a chain of H / 256 memory round trips; one
// expert a wave makes them 128 whose loads go out at once (H = 2048, E = 128: 16 tokens 11.8 -> 6.4 us, 128 tokens
// 11.4 -> 10.7; at 512 the activations would be read 128 times).
template <int CQ, int EW>
__global__ __launch_bounds__(256) void k_moe_logits(const float *__restrict__ x, const float *__restrict__ wr,
                                                    float *__restrict__ logits, int T, int H, int E,
                                                    int8_t *__restrict__ qx, float *__restrict__ sx)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int t0 = blockIdx.x * 16 + wave * 4;
    const int e0 = blockIdx.y * EW;

    // the token row this wave quantizes (if any) is requested first: its loads then fly under the logits' rounds
    // instead of costing a memory round trip after them
    constexpr int LPB = 16;
    constexpr int CQR = CQ > 0 ? CQ : 1;
    const int jq = lane % LPB, nchunk = H / 8;
    const int qtt = (int)blockIdx.y * 4 + wave;                 // the workgroups of a token group deal its 16 rows
    const int qrow = blockIdx.x * 16 + qtt;
    const bool has_row = CQ > 0 && qtt < 16 && qrow < T;        // whole wave
    float v[CQR][8];
    int base[CQR];
    if constexpr (CQ > 0) {
        const float *xrow = x + (int64_t)min(qrow, T - 1) * H;
#pragma unroll
        for (int i = 0; i < CQ; ++i) {
            const int c = lane + i * 64;
            base[i] = (c / LPB) * 128 + 4 * jq;
            if (has_row && c < nchunk) {
                const float4 lo = *reinterpret_cast<const float4 *>(xrow + base[i]);
                const float4 hi = *reinterpret_cast<const float4 *>(xrow + base[i] + 64);
                v[i][0] = lo.x; v[i][1] = lo.y; v[i][2] = lo.z; v[i][3] = lo.w;
                v[i][4] = hi.x; v[i][5] = hi.y; v[i][6] = hi.z; v[i][7] = hi.w;
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[i][e] = 0.0f;
            }
        }
    }

    float p[4 * EW];
#pragma unroll
    for (int i = 0; i < 4 * EW; ++i) p[i] = 0.0f;
    const float *xr[4];
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) xr[tt] = x + (int64_t)min(t0 + tt, T - 1) * H + 4 * lane;
    const float *wp = wr + (int64_t)e0 * H + 4 * lane;
    // Eight experts at a time: while the 128 FMAs of one half run, the weights of the next half (and, behind a
    // second half, the token rows of the next round) are already on their way; with one wave per SIMD the loop is
    // otherwise a chain of memory round trips.  Every dot product still takes its terms in the same order.
    const int nj = H / 256;
    if constexpr (EW == 16) {
        float4 xv[4], xn[4], wa[8], wb[8];
    #pragma unroll
        for (int tt = 0; tt < 4; ++tt) xv[tt] = *reinterpret_cast<const float4 *>(xr[tt]);
    #pragma unroll
        for (int e = 0; e < 8; ++e) wa[e] = *reinterpret_cast<const float4 *>(wp + (int64_t)e * H);
        for (int j = 0; j < nj; ++j) {
    #pragma unroll
            for (int e = 0; e < 8; ++e) wb[e] = *reinterpret_cast<const float4 *>(wp + (int64_t)(8 + e) * H + 256 * j);
    #pragma unroll
            for (int tt = 0; tt < 4; ++tt)
    #pragma unroll
                for (int e = 0; e < 8; ++e) {
                    float a = p[tt * 16 + e];
                    a = __builtin_fmaf(xv[tt].x, wa[e].x, a);
                    a = __builtin_fmaf(xv[tt].y, wa[e].y, a);
                    a = __builtin_fmaf(xv[tt].z, wa[e].z, a);
                    a = __builtin_fmaf(xv[tt].w, wa[e].w, a);
                    p[tt * 16 + e] = a;
                }
            const int jn = min(j + 1, nj - 1);   // (the last round fetches itself again: no branch around loads)
    #pragma unroll
            for (int e = 0; e < 8; ++e) wa[e] = *reinterpret_cast<const float4 *>(wp + (int64_t)e * H + 256 * jn);
    #pragma unroll
            for (int tt = 0; tt < 4; ++tt) xn[tt] = *reinterpret_cast<const float4 *>(xr[tt] + 256 * jn);
    #pragma unroll
            for (int tt = 0; tt < 4; ++tt)
    #pragma unroll
                for (int e = 0; e < 8; ++e) {
                    float a = p[tt * 16 + 8 + e];
                    a = __builtin_fmaf(xv[tt].x, wb[e].x, a);
                    a = __builtin_fmaf(xv[tt].y, wb[e].y, a);
                    a = __builtin_fmaf(xv[tt].z, wb[e].z, a);
                    a = __builtin_fmaf(xv[tt].w, wb[e].w, a);
                    p[tt * 16 + 8 + e] = a;
                }
    #pragma unroll
            for (int tt = 0; tt < 4; ++tt) xv[tt] = xn[tt];
        }
    } else if constexpr (EW == 1) {
        // few tokens: one expert a wave and JB rounds' loads requested at a time, the next JB behind them, so that rows of
        // up to 2048 floats are in flight as a whole before the first FMA
        constexpr int JB = 4;
        float4 xa[2][JB][4], wa[2][JB];
        auto request = [&](int set, int j0) {
#pragma unroll
            for (int u = 0; u < JB; ++u) {
                const int j = min(j0 + u, nj - 1);
                wa[set][u] = *reinterpret_cast<const float4 *>(wp + 256 * j);
#pragma unroll
                for (int tt = 0; tt < 4; ++tt) xa[set][u][tt] = *reinterpret_cast<const float4 *>(xr[tt] + 256 * j);
            }
        };
        auto add = [&](int set, int j0) {
#pragma unroll
            for (int u = 0; u < JB; ++u) {
                if (j0 + u >= nj) break;   // (uniform)
                const float4 w = wa[set][u];
#pragma unroll
                for (int tt = 0; tt < 4; ++tt) {
                    const float4 v = xa[set][u][tt];
                    float a = p[tt];
                    a = __builtin_fmaf(v.x, w.x, a);
                    a = __builtin_fmaf(v.y, w.y, a);
                    a = __builtin_fmaf(v.z, w.z, a);
                    a = __builtin_fmaf(v.w, w.w, a);
                    p[tt] = a;
                }
            }
        };
        if (t0 < T) {   // whole wave
            request(0, 0);
            for (int j = 0; j < nj; j += 2 * JB) {
                request(1, j + JB);
                add(0, j);
                if (j + 2 * JB < nj) request(0, j + 2 * JB);
                add(1, j + JB);
            }
        }
    } else {
        // one group of eight experts: the next round's weights and token rows are requested before this round's
        // 128 FMAs
        float4 xv[4], xn[4], wa[8], wn[8];
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) xv[tt] = *reinterpret_cast<const float4 *>(xr[tt]);
#pragma unroll
        for (int e = 0; e < 8; ++e) wa[e] = *reinterpret_cast<const float4 *>(wp + (int64_t)e * H);
        for (int j = 0; j < nj; ++j) {
            const int jn = min(j + 1, nj - 1);   // (the last round fetches itself again: no branch around loads)
#pragma unroll
            for (int e = 0; e < 8; ++e) wn[e] = *reinterpret_cast<const float4 *>(wp + (int64_t)e * H + 256 * jn);
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) xn[tt] = *reinterpret_cast<const float4 *>(xr[tt] + 256 * jn);
#pragma unroll
            for (int tt = 0; tt < 4; ++tt)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    float a = p[tt * 8 + e];
                    a = __builtin_fmaf(xv[tt].x, wa[e].x, a);
                    a = __builtin_fmaf(xv[tt].y, wa[e].y, a);
                    a = __builtin_fmaf(xv[tt].z, wa[e].z, a);
                    a = __builtin_fmaf(xv[tt].w, wa[e].w, a);
                    p[tt * 8 + e] = a;
                }
#pragma unroll
            for (int e = 0; e < 8; ++e) wa[e] = wn[e];
#pragma unroll
            for (int tt = 0; tt < 4; ++tt) xv[tt] = xn[tt];
        }
    }
    if constexpr (EW == 16) {
        fold<32, 32>(p, lane);
        fold<16, 16>(p, lane);
        fold<8, 8>(p, lane);
        fold<4, 4>(p, lane);
        fold<2, 2>(p, lane);
        fold<1, 1>(p, lane);
        // lane l now holds pair l: token l/16, expert e0 + l%16
        const int t = t0 + (lane >> 4);
        if (t < T) logits[(int64_t)t * E + e0 + (lane & 15)] = p[0];
    } else if constexpr (EW == 1) {
        fold<32, 2>(p, lane);
        fold<16, 1>(p, lane);
        p[0] = add_lane<1>(add_lane<2>(add_lane<4>(add_lane<8>(p[0]))));
        const int t = t0 + (lane >> 4);   // the 16 lanes of a group hold the same token's sum
        if ((lane & 15) == 0 && t < T) logits[(int64_t)t * E + e0] = p[0];
    } else {
        static_assert(EW == 8, "experts per wave");
#pragma unroll
        for (int i = 0; i < 32; ++i) p[i] = add_lane<32>(p[i]);
        fold<16, 16>(p, lane);
        fold<8, 8>(p, lane);
        fold<4, 4>(p, lane);
        fold<2, 2>(p, lane);
        fold<1, 1>(p, lane);
        // lanes l and l ^ 32 now hold pair l % 32: token (l % 32) / 8, expert e0 + l % 8
        const int t = t0 + ((lane & 31) >> 3);
        if (lane < 32 && t < T) logits[(int64_t)t * E + e0 + (lane & 7)] = p[0];
    }
    if constexpr (CQ > 0) {
        if (has_row) {
            float amax = 0.0f;
#pragma unroll
            for (int i = 0; i < CQ; ++i) {
                fwht_codes<128>(v[i], jq);
                amax = fmaxf(amax, abs8(v[i]));
            }
            amax = max_lanes<64>(amax);
            const float sc = (amax == 0.0f) ? 1.0f : amax / 127.0f;
            const float inv = (amax == 0.0f) ? 0.0f : 127.0f / amax;
            if (lane == 0) sx[qrow] = sc;
            int8_t *qr = qx + (int64_t)qrow * H;
#pragma unroll
            for (int i = 0; i < CQ; ++i) {
                if (lane + i * 64 < nchunk) {
                    *reinterpret_cast<uint32_t *>(qr + base[i]) = quant4(v[i][0], v[i][1], v[i][2], v[i][3], inv);
                    *reinterpret_cast<uint32_t *>(qr + base[i] + 64) = quant4(v[i][4], v[i][5], v[i][6], v[i][7], inv);
                }
            }
        }
        // fewer than four expert groups: a wave has further rows of the token group to do
        for (int tt = qtt + (int)gridDim.y * 4; tt < 16; tt += (int)gridDim.y * 4) {
            const int row = blockIdx.x * 16 + tt;
            if (row >= T) break;   // whole wave
            const float *xrow = x + (int64_t)row * H;
#pragma unroll
            for (int i = 0; i < CQ; ++i) {
                if (lane + i * 64 < nchunk) {
                    const float4 lo = *reinterpret_cast<const float4 *>(xrow + base[i]);
                    const float4 hi = *reinterpret_cast<const float4 *>(xrow + base[i] + 64);
                    v[i][0] = lo.x; v[i][1] = lo.y; v[i][2] = lo.z; v[i][3] = lo.w;
                    v[i][4] = hi.x; v[i][5] = hi.y; v[i][6] = hi.z; v[i][7] = hi.w;
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[i][e] = 0.0f;
                }
            }
            float amax = 0.0f;
#pragma unroll
            for (int i = 0; i < CQ; ++i) {
                fwht_codes<128>(v[i], jq);
                amax = fmaxf(amax, abs8(v[i]));
            }
            amax = max_lanes<64>(amax);
            const float sc = (amax == 0.0f) ? 1.0f : amax / 127.0f;
            const float inv = (amax == 0.0f) ? 0.0f : 127.0f / amax;
            if (lane == 0) sx[row] = sc;
            int8_t *qr = qx + (int64_t)row * H;
#pragma unroll
            for (int i = 0; i < CQ; ++i) {
                if (lane + i * 64 < nchunk) {
                    *reinterpret_cast<uint32_t *>(qr + base[i]) = quant4(v[i][0], v[i][1], v[i][2], v[i][3], inv);
                    *reinterpret_cast<uint32_t *>(qr + base[i] + 64) = quant4(v[i][4], v[i][5], v[i][6], v[i][7], inv);
                }
            }
        }
    }
}

template <int CTRL>
__device__ __forceinline__ float dpp_f(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float readlane_f(float v, int l)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}

// one wave per token: k rounds of (wave-wide max, lowest index among the lanes that hold it); lane l holds
// experts l, l+64, l+128, l+192.  Ties go to the lower expert index; picks come out by descending logit.
// Lane s < topk returns pick s and leaves its weight in weight.  U: the slots of 64 experts that there are.
// The loop is one serial chain, so a slot less is a link less: the layer with four slots always and the picks' values in
// an array of registers, before -> after: 1 token 37.9 -> 37.3 us, 16 tokens 110.1 -> 109.4, 16 of 64 experts 58.4 -> 57.6.
template <int U>
__device__ __forceinline__ int topk_row(const float *__restrict__ logits, int t, int E, int topk, int lane, float &weight)
{
    float mine[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int i = lane + 64 * u;
        mine[u] = i < E ? logits[(int64_t)t * E + i] : -INFINITY;
    }
    float first = 0.0f, mine_top = 0.0f;   // of pick 0; of pick "lane"
    int pick_lane = 0;                     // lane s keeps pick s
    for (int s = 0; s < topk; ++s) {
        // wave-wide maximum: four DPP steps leave every 16-lane row with its own maximum, four scalar reads join the
        // rows (a chain of cross-lane permutes costs five times as many cycles, and this loop is all latency)
        float v = -INFINITY;               // also what a row of nothing but NaN gives
#pragma unroll
        for (int u = 0; u < U; ++u) v = fmaxf(v, mine[u]);
        v = fmaxf(v, dpp_f<0xB1>(v));    // quad_perm [1,0,3,2]
        v = fmaxf(v, dpp_f<0x4E>(v));    // quad_perm [2,3,0,1]
        v = fmaxf(v, dpp_f<0x124>(v));   // row_ror:4
        v = fmaxf(v, dpp_f<0x128>(v));   // row_ror:8
        v = fmaxf(fmaxf(readlane_f(v, 0), readlane_f(v, 16)), fmaxf(readlane_f(v, 32), readlane_f(v, 48)));
        // lowest expert index holding v: experts of slot u are 64u .. 64u+63, so the first non-empty ballot wins
        int win = -1;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const unsigned long long bal = __ballot(mine[u] == v);
            if (win < 0 && bal) {
                const int wl = __ffsll((long long)bal) - 1;
                win = wl + 64 * u;
                if (lane == wl) mine[u] = -INFINITY;   // taken
            }
        }
        if (win < 0 && U < 4) win = 64 * U;   // a row of nothing but NaN: an expert that is not there, which the dispatch skips
        if (s == 0) first = v;
        if (lane == s) pick_lane = win, mine_top = v;
    }
    // lane s evaluates e_s = expf(l_s - l_0) once; the sum runs over the picks in pick order, as the oracle's does
    const float e = lane < topk ? expf(mine_top - first) : 0.0f;
    float sum = 0.0f;
#pragma unroll
    for (int q = 0; q < MAX_TOPK; ++q)
        if (q < topk) sum = sum + readlane_f(e, q);
    weight = e / sum;
    return pick_lane;
}

__device__ __forceinline__ int topk_row(const float *__restrict__ logits, int t, int E, int topk, int lane, float &weight)
{
    return E <= 64    ? topk_row<1>(logits, t, E, topk, lane, weight)
           : E <= 128 ? topk_row<2>(logits, t, E, topk, lane, weight)
                      : topk_row<4>(logits, t, E, topk, lane, weight);
}

__global__ __launch_bounds__(256) void k_moe_topk(const float *__restrict__ logits, int32_t *__restrict__ idx,
                                                  float *__restrict__ w, int T, int E, int topk)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int t = blockIdx.x * 4 + wave;
    if (t >= T) return;   // whole wave
    float weight;
    const int pick = topk_row(logits, t, E, topk, lane, weight);
    if (lane < topk) {
        idx[(int64_t)t * topk + lane] = pick;
        w[(int64_t)t * topk + lane] = weight;
    }
}

// Inclusive sum over the lanes up to this one, on the vector pipe alone (a shuffle would cost an LDS round trip a step).
__device__ __forceinline__ int wave_scan(int v)
{
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);    // row_shr:1, 2, 4, 8
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);   // row_bcast:15 into rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);   // row_bcast:31 into rows 2 and 3
    return v;
}

// -------------------------------------------------------------- a10 dispatch
// One workgroup.  bm[t/32][e] bit t%32 = "token t picked expert e" (a token
// picks an expert at most once), so the stable rank of pair (t, slot) inside
// its expert is the number of set bits below t in column e.
// One chain of latencies on one compute unit, so instructions count: a division by topk is a multiplication (magic, see
// topk_magic), neighbouring lanes read neighbouring words, and eight of them are requested at a
// time.  us by itself in a chain, 128 experts, before -> after: 512 tokens 6.5 -> 4.9, 2048 tokens 30.2 -> 15.0, 16 and 64 tokens 3.0.
__device__ __forceinline__ void dispatch_pairs(uint32_t *s_dyn, const int32_t *idx, int32_t *__restrict__ perm,
                                               int32_t *__restrict__ seg_off, int T, int E, int topk, uint32_t magic)
{
    const int W = (T + 31) >> 5;
    uint32_t *bm = s_dyn;                 // [W][E]
    uint32_t *pre = s_dyn + E * W;        // [W][E] exclusive popcount prefix
    int *seg = reinterpret_cast<int *>(s_dyn + 2 * E * W);  // [E+1]
    const int tid = threadIdx.x, nt = blockDim.x;
    const int P = T * topk;
    const auto token = [&](int pr) { return magic ? (int)__umulhi((uint32_t)pr, magic) : pr / topk; };
    for (int i = tid; i < E * W; i += nt) bm[i] = 0u;
    // a thread's pairs stay in registers between the two passes when they are few (one global round trip less)
    constexpr int KEEP = 8;
    const bool keep = P <= KEEP * nt;
    int mine[KEEP];
    if (keep) {
#pragma unroll
        for (int i = 0; i < KEEP; ++i) {
            const int pr = tid + i * nt;
            mine[i] = pr < P ? idx[pr] : -1;
        }
    }
    __syncthreads();
    if (keep) {
#pragma unroll
        for (int i = 0; i < KEEP; ++i) {
            const int e = mine[i], t = token(tid + i * nt);
            if (e >= 0 && e < E) atomicOr(&bm[(t >> 5) * E + e], 1u << (t & 31));
        }
    } else {
        for (int pr = tid; pr < P; pr += nt) {
            const int e = idx[pr], t = token(pr);
            if (e >= 0 && e < E) atomicOr(&bm[(t >> 5) * E + e], 1u << (t & 31));
        }
    }
    __syncthreads();
    for (int e = tid; e < E; e += nt) {
        int c = 0;
        for (int w0 = 0; w0 < W; w0 += 8) {
            uint32_t b[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) b[i] = bm[min(w0 + i, W - 1) * E + e];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                if (w0 + i >= W) break;
                pre[(w0 + i) * E + e] = (uint32_t)c;
                c += __popc(b[i]);
            }
        }
        seg[e + 1] = c;
    }
    __syncthreads();
    // exclusive scan of the E counts by one wave: lane l sums its run of ceil(E/64) counts, the wave scans the 64
    // run totals, the lane writes its run back (a serial loop over E through LDS costs a dependent
    // LDS round trip per expert)
    if (tid < 64) {
        const int run = (E + 63) / 64;
        const int lo = min(tid * run, E), hi = min(lo + run, E);
        int sum = 0;
        for (int e = lo; e < hi; ++e) sum += seg[e + 1];
        int acc = wave_scan(sum) - sum;
        if (tid == 0) seg[0] = 0;
        for (int e = lo; e < hi; ++e) {
            acc += seg[e + 1];
            seg[e + 1] = acc;
        }
    }
    __syncthreads();
    for (int e = tid; e <= E; e += nt) seg_off[e] = seg[e];
    if (keep) {
#pragma unroll
        for (int i = 0; i < KEEP; ++i) {
            const int pr = tid + i * nt;
            const int e = mine[i], t = token(pr);
            if (e < 0 || e >= E) continue;
            const uint32_t word = bm[(t >> 5) * E + e];
            const int pos = seg[e] + (int)pre[(t >> 5) * E + e] + __popc(word & ((1u << (t & 31)) - 1u));
            perm[pos] = pr;
        }
    } else {
        for (int pr = tid; pr < P; pr += nt) {
            const int e = idx[pr], t = token(pr);
            if (e < 0 || e >= E) continue;
            const uint32_t word = bm[(t >> 5) * E + e];
            const int pos = seg[e] + (int)pre[(t >> 5) * E + e] + __popc(word & ((1u << (t & 31)) - 1u));
            perm[pos] = pr;
        }
    }
}

__global__ __launch_bounds__(1024) void k_moe_dispatch(const int32_t *__restrict__ idx, int32_t *__restrict__ perm,
                                                       int32_t *__restrict__ seg_off, int T, int E, int topk, uint32_t magic)
{
    extern __shared__ uint32_t s_dyn[];
    dispatch_pairs(s_dyn, idx, perm, seg_off, T, E, topk, magic);
}

// Top-k and dispatch of few tokens in one launch: a wave a token, the picks go to the dispatch
// through LDS.  Both kernels are all latency (a launch of 4 to 5 us for a few hundred bytes), so one of the two is saved;
// the layer's time, two launches -> one: 1 token of 128 experts 37.3 -> 36.4 us, 4 tokens 47.7 -> 46.8, 16 tokens 109.5 -> 109.1,
// 16 of 64 experts 57.6 -> 57.0.  Beyond a token a wave the one workgroup's rounds cost more than the launch: 32 tokens
// 123.9 -> 126.0 us, 64 tokens 138.2 -> 146.6.
constexpr int64_t ROUTE_DISPATCH_MAX_T = 16;
__global__ __launch_bounds__(1024) void k_moe_topk_dispatch(const float *__restrict__ logits, int32_t *__restrict__ idx,
                                                            float *__restrict__ w, int32_t *__restrict__ perm,
                                                            int32_t *__restrict__ seg_off, int T, int E, int topk, uint32_t magic)
{
    __shared__ int32_t s_idx[ROUTE_DISPATCH_MAX_T * MAX_TOPK];
    extern __shared__ uint32_t s_dyn[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (const int t = wave; t < T) {   // one token a wave
        float weight;
        const int pick = topk_row(logits, t, E, topk, lane, weight);
        if (lane < topk) {
            s_idx[t * topk + lane] = pick;
            idx[t * topk + lane] = pick;
            w[t * topk + lane] = weight;
        }
    }
    __syncthreads();
    dispatch_pairs(s_dyn, s_idx, perm, seg_off, T, E, topk, magic);
}

// ------------------------------------------------------- a11 grouped GEMMs
// One kernel for both expert contractions.  A workgroup of 4 waves owns two groups of 16 weight rows of one
// expert (gate/up: rows n0.. of wg and the same rows of wu, so SwiGLU happens in the epilogue; down: rows
// n0.. and n0+16.. of wd) and walks the expert's tokens 32 at a time.  Waves split K.  Every wave streams
// its K slice through a private ring of LDS stages filled by direct-to-LDS loads of 8 rows x 128 bytes
// (weights and gathered activation rows alike; a load shaped like an MFMA fragment, 16 rows x 64 bytes, runs
// at a third of the bandwidth), XOR-swizzled so that the v_mfma_i32_16x16x64_i8 fragment reads are conflict
// free.  No barrier inside the stream; partial accumulators of the four waves meet in LDS.
constexpr int MT = 2;             // 16-token fragments per pass
constexpr int NGRP = 2;           // 16-row weight groups per workgroup
constexpr int RING = 2;           // stages per wave
constexpr int BLK = 2 * (NGRP + MT);
constexpr int STAGE_BYTES = BLK * 1024;
constexpr int RING_BYTES = 4 * RING * STAGE_BYTES;
constexpr int EXPERT_LDS = RING_BYTES + 4 * NGRP * MT * 4 * 64 * 4;

template <bool DOWN>
__global__ __launch_bounds__(256) void k_moe_expert_gemm(const int8_t *__restrict__ act,
                                                         const float *__restrict__ act_scale,
                                                         const int32_t *__restrict__ perm,
                                                         const int32_t *__restrict__ seg_off,
                                                         const int8_t *__restrict__ w0, const float *__restrict__ sc0,
                                                         const int8_t *__restrict__ w1, const float *__restrict__ sc1,
                                                         float *__restrict__ out, int Kdim, int Nrows, int Hout,
                                                         int topk, int nch)
{
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int e = blockIdx.y;
    const int seg0 = seg_off[e], count = seg_off[e + 1] - seg0;
    if (count <= 0) return;
    // gate/up: the 4 waves split K (2048 bytes = 16 steps).  down: K is short (768 bytes = 6 steps), so each
    // wave takes its own 32 rows over the whole of K and nothing has to be added across waves
    // A workgroup walks `nch` consecutive row chunks (16 rows for gate/up, 128 for down) as ONE stream: the
    // loads of the next chunk are already in flight while the partial sums of this one are added and stored,
    // and the segment / permutation lookups are paid once per workgroup.
    constexpr int CHUNK_ROWS = DOWN ? 128 : 16;
    const int n0 = DOWN ? blockIdx.x * nch * 128 + wave * 32 : blockIdx.x * nch * 16;
    char *ring = smem + wave * (RING * STAGE_BYTES);
    int *s_part = reinterpret_cast<int *>(smem + RING_BYTES);   // [4 waves][NGRP][MT][4][64]

    // load side: lane l = 8*rho + c fetches chunk c ^ sigma(rho, block parity) of row rho of the block
    const int rho = lane >> 3, c8 = lane & 7;
    const int8_t *wsrc[2 * NGRP];
#pragma unroll
    for (int b = 0; b < 2 * NGRP; ++b) {
        const int sigma = ((b & 1) << 2) | (rho >> 1);
        const int grp = b >> 1;
        int rowi = n0 + (DOWN ? grp * 16 : 0) + (b & 1) * 8 + rho;
        if (rowi > Nrows - 1) rowi = Nrows - 1;
        const int8_t *base = (DOWN || grp == 0) ? w0 : w1;
        wsrc[b] = base + ((int64_t)e * Nrows + rowi) * Kdim + ((c8 ^ sigma) << 4);
    }
    const int steps = Kdim >> 7;
    const int s0 = DOWN ? 0 : steps * wave / 4, s1 = DOWN ? steps : steps * (wave + 1) / 4;

    // read side: fragment (16-row group, K half kk): lane (r = l%16, g = l/16) reads row r, chunk 4*kk + g
    const int r = lane & 15, g_ = lane >> 4;
    int roff[2];
    {
        const int rr = r & 7, bpar = r >> 3;
        const int sigma = (bpar << 2) | (rr >> 1);
        roff[0] = bpar * 1024 + ((8 * rr + ((0 + g_) ^ sigma)) << 4);
        roff[1] = bpar * 1024 + ((8 * rr + ((4 + g_) ^ sigma)) << 4);
    }

    for (int base = 0; base < count; base += 16 * MT) {
        // gathered activation rows of this pass (rows past the segment repeat its last row and are never stored)
        const int8_t *xsrc[2 * MT];
#pragma unroll
        for (int b = 0; b < 2 * MT; ++b) {
            const int sigma = ((b & 1) << 2) | (rho >> 1);
            const int pos = seg0 + min(base + b * 8 + rho, count - 1);
            const int64_t arow = DOWN ? (int64_t)pos : (int64_t)(perm[pos] / topk);
            xsrc[b] = act + arow * Kdim + ((c8 ^ sigma) << 4);
        }
        const int nsw = s1 - s0;            // K steps of this wave per chunk
        const int total_f = nch * nsw;      // flattened (chunk, step) stages of this wave
        auto issue = [&](int slot, int f) {
            const int fc = f < total_f ? f : total_f - 1;   // past the end: re-fetch the last stage (uniform vmcnt arithmetic)
            const int ch = fc / nsw, st = s0 + (fc - ch * nsw);
            char *sb = ring + slot * STAGE_BYTES;
            const int64_t koff = (int64_t)st * 128;
            const int64_t woff = (int64_t)ch * CHUNK_ROWS * Kdim + koff;
#pragma unroll
            for (int b = 0; b < 2 * NGRP; ++b)
                __builtin_amdgcn_global_load_lds((gptr_t)(wsrc[b] + woff), (lptr_t)(sb + b * 1024), 16, 0, 0);
#pragma unroll
            for (int b = 0; b < 2 * MT; ++b)
                __builtin_amdgcn_global_load_lds((gptr_t)(xsrc[b] + koff), (lptr_t)(sb + (2 * NGRP + b) * 1024), 16, 0, 0);
        };
        if (nsw > 0) {
#pragma unroll
            for (int d = 0; d < RING; ++d) issue(d, d);
        }
        int slot = 0, f = 0;
        for (int ch = 0; ch < nch; ++ch) {
        const int nc0 = n0 + ch * CHUNK_ROWS;
        v4i acc[NGRP][MT];
#pragma unroll
        for (int a = 0; a < NGRP; ++a)
#pragma unroll
            for (int b = 0; b < MT; ++b) acc[a][b] = (v4i){0, 0, 0, 0};
        for (int i = 0; i < nsw; ++i, ++f) {
            wait_vm<(RING - 1) * BLK>();   // the oldest stage in flight has landed
            const char *sb = ring + slot * STAGE_BYTES;
            v4i wf[NGRP][2], xf[MT][2];
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
                for (int a = 0; a < NGRP; ++a) wf[a][kk] = *reinterpret_cast<const v4i *>(sb + a * 2048 + roff[kk]);
#pragma unroll
                for (int b = 0; b < MT; ++b) xf[b][kk] = *reinterpret_cast<const v4i *>(sb + (NGRP + b) * 2048 + roff[kk]);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // fragments are in registers: the slot may be refilled
            issue(slot, f + RING);
#pragma unroll
            for (int kk = 0; kk < 2; ++kk)
#pragma unroll
                for (int a = 0; a < NGRP; ++a)
#pragma unroll
                    for (int b = 0; b < MT; ++b)
                        acc[a][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[a][kk], xf[b][kk], acc[a][b], 0, 0, 0);
            slot = slot + 1 == RING ? 0 : slot + 1;
        }
        __syncthreads();   // the previous chunk's epilogue has finished reading s_part
#pragma unroll
        for (int a = 0; a < NGRP; ++a)
#pragma unroll
            for (int b = 0; b < MT; ++b)
#pragma unroll
                for (int q = 0; q < 4; ++q) s_part[(((wave * NGRP + a) * MT + b) * 4 + q) * 64 + lane] = acc[a][b][q];
        __syncthreads();
        // accumulator layout: lane l, register q  <->  weight row 4*(l/16)+q, token l%16
        auto total = [&](int a, int row, int nn) {
            const int b = row >> 4, src = (nn >> 2) * 16 + (row & 15), q = nn & 3;
            int sum = 0;
#pragma unroll
            for (int wv = 0; wv < 4; ++wv) sum += s_part[(((wv * NGRP + a) * MT + b) * 4 + q) * 64 + src];
            return sum;
        };
        auto own = [&](int wv, int a, int row, int nn) {   // down: one wave's accumulator is already the total
            const int b = row >> 4, src = (nn >> 2) * 16 + (row & 15), q = nn & 3;
            return s_part[(((wv * NGRP + a) * MT + b) * 4 + q) * 64 + src];
        };
        if constexpr (!DOWN) {
            // 32 tokens x 16 channels, channel fastest; h = silu(g) * u in sorted-pair order
            for (int o = tid; o < 16 * MT * 16; o += 256) {
                const int nl = o & 15, row = o >> 4;
                if (base + row >= count || nc0 + nl >= Nrows) continue;
                const int pos = seg0 + base + row;
                const float sxt = act_scale[perm[pos] / topk];
                const float gv = ((float)total(0, row, nl) * sxt) * sc0[(int64_t)e * Nrows + nc0 + nl];
                const float uv = ((float)total(1, row, nl) * sxt) * sc1[(int64_t)e * Nrows + nc0 + nl];
                out[(int64_t)pos * Nrows + nc0 + nl] = silu(gv) * uv;
            }
        } else {
            // 32 tokens x 128 channels (32 per wave); out[pair] in pair order, channel fastest
            const int nbase = (blockIdx.x * nch + ch) * 128;
            for (int o = tid; o < 16 * MT * 128; o += 256) {
                const int nl = o & 127, row = o >> 7;
                if (base + row >= count || nbase + nl >= Nrows) continue;
                const int pos = seg0 + base + row;
                const int sum = own(nl >> 5, (nl >> 4) & 1, row, nl & 15);
                out[(int64_t)perm[pos] * Hout + nbase + nl] =
                    ((float)sum * act_scale[pos]) * sc0[(int64_t)e * Nrows + nbase + nl];
            }
        }
        }   // chunks
        wait_vm<0>();   // trailing re-fetches must not write LDS after the workgroup has gone
    }
}

// The same contraction with the activation fragments held in registers (possible when a wave's K slice is at
// most NSMAX steps of 128 bytes): only weights travel through the ring, twice as many of them are in flight
// for the same LDS, and a workgroup walks several row chunks against one set of activation registers.
// Its direct-to-LDS loads are asm statements: in front of an LDS atomic the compiler waits for every one in flight that it knows of.
// Stages in flight per wave.  The down kernel by itself, traced at 512 tokens and a router's own counts, takes 59.1 us with four,
// 58.5 with three, 57.6 with two; the layer that it is part of 186.5, 187.0 and 188.4 (with two, 3 % less to 1 % more elsewhere).
constexpr int RX_RING = 4;
constexpr int RX_STAGE = 2 * NGRP * 1024;
constexpr int RX_RING_BYTES = 4 * RX_RING * RX_STAGE;
constexpr int RX_MT = 4;   // most 16-token fragments per pass
constexpr int RX_RED_BYTES = NGRP * RX_MT * 4 * 64 * 4;
constexpr int RX_SCALES = 1024;   // weight scales of a run of chunks: four for each of 256 threads
constexpr int rx_most_chunks(bool down) { return RX_SCALES / (down ? 128 : 32); }   // of a run
constexpr int RX_LDS = RX_RING_BYTES + RX_RED_BYTES + 16 * RX_MT * 8 + RX_SCALES * 4;   // 8 bytes of metadata a token
static_assert(2 * RX_LDS <= 160 * 1024, "two workgroups a unit");

// Most tokens of a pass over an expert's weights: what the registers hold.  (512 tokens, H = 2048, 12 of 128 experts with more
// than 48: 180 us for the layer's FFN with passes of 48, 176 with 64.)
constexpr int rx_most(int nsmax) { return nsmax > 6 ? 32 : nsmax > 4 ? 48 : 64; }

// Where the down kernel makes the codes of its rows itself (OWN) and the quantizer's launch between the two expert kernels goes.
// Every workgroup of an expert makes all of its codes, at 0.8 us for each row of a wave (some 330 vector instructions, one wave a
// SIMD), so what it costs is the rows of the fullest expert.  The host does not know them: at most T, and that many where all tokens
// go to the same experts.  FFN, us with the launch -> without, top-8 of 128, H = 2048, I = 768: 16 tokens one to an expert 121.5 ->
// 119.4, as a router sends them 94.2 -> 91.6, half of them to the same eight 68.1 -> 66.9, all of them 29.5 -> 30.8; 8 tokens to the
// same eight 28.1 -> 27.6; top-4 of 64, H = 1024, I = 512, the four of 16 tokens 35.0 -> 32.9, 32.2 -> 29.7, 27.1 -> 26.4, 21.1 -> 20.9;
// 1 token 26.1 -> 25.1 and 18.9 -> 17.1.  Beyond 16 tokens the rows of one expert can cost more than a launch: 24 tokens 104.0 -> 101.8 as
// a router sends them, 32.2 -> 34.7 all to the same; 32 tokens 117.3 -> 114.5 and 33.2 -> 38.1.  And so with few experts: 16 of them, H =
// 1024, I = 256, 8 rows an expert 28.0 -> 26.3, 12 rows an expert 43.4 -> 45.4.
constexpr int OWN_PASS = 16;
static bool own_codes(int64_t T, int64_t E, int topk) { return T <= OWN_PASS && T * topk <= 8 * E; }

// (the compiler does not see that a pointer out of an asm statement is one to device memory)
template <typename T>
using global_ptr = __attribute__((address_space(1))) T *;

// One pass: at most 16 * MTT of an expert's pairs (from pos0 on, n of them) against nch row chunks from chunk c0 on.
// first: the workgroup's first pass over these chunks, which brings their weight scales.
// OWN (down, see own_codes): the pairs' codes are made here, from fp32 rows h; the workgroup with the expert's first
// chunk leaves them in act and act_scale.
template <bool DOWN, int NSMAX, int MTT, bool OWN>
__device__ __forceinline__ void rx_pass(char *smem, int8_t *act, float *act_scale, const float *__restrict__ h,
                                        const int32_t *__restrict__ perm, const int8_t *__restrict__ w0,
                                        const float *__restrict__ sc0, const int8_t *__restrict__ w1,
                                        const float *__restrict__ sc1, float *__restrict__ out, int Kdim, int Nrows, int topk,
                                        int e, int c0, int nch, int pos0, int n, bool first)
{
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // gate/up: the 4 waves split K (2048 bytes = 16 steps).  down: K is short (768 bytes = 6 steps), so each
    // wave takes its own 32 rows over the whole of K and nothing has to be added across waves.
    // The row chunks (16 gate and 16 up rows, or 128 down rows) are ONE stream: the loads of the next chunk are already
    // in flight while the partial sums of this one are added and stored.
    constexpr int CHUNK_ROWS = DOWN ? 128 : 16, SCW = DOWN ? 128 : 32;
    constexpr int RING = RX_RING;
    char *ring = smem + wave * (RING * RX_STAGE);
    int *s_red = reinterpret_cast<int *>(smem + RX_RING_BYTES);    // [NGRP][MTT][4][64] sums over the four K slices (gate/up)
    // token metadata and the chunks' weight scales sit in LDS so that the epilogue of a chunk issues no dependent global
    // loads (each would cost a memory round trip per chunk)
    int *s_dst = reinterpret_cast<int *>(smem + RX_RING_BYTES + RX_RED_BYTES);            // [16 RX_MT] output row
    float *s_tsc = reinterpret_cast<float *>(s_dst + 16 * RX_MT);                                // [16 RX_MT] token scale
    float *s_wsc = s_tsc + 16 * RX_MT;                                                           // [nch][SCW]

    __syncthreads();   // the previous pass has finished with the token metadata and the scales, and every ring is idle

    // load side: lane l = 8*rho + c8 fetches chunk c8 ^ sigma(rho, block parity) of row rho of a block of 8 rows
    const int rho = lane >> 3, c8 = lane & 7;
    const int steps = Kdim >> 7;
    const int s0 = DOWN ? 0 : steps * wave / 4;
    const int nsw = (DOWN ? steps : steps * (wave + 1) / 4) - s0;   // K steps of this wave per chunk (<= NSMAX)
    const unsigned woff0 = (unsigned)rho * (unsigned)Kdim + ((c8 ^ (rho >> 1)) << 4);   // an even block; an odd one is below it
    const unsigned woff1 = (unsigned)(8 + rho) * (unsigned)Kdim + ((c8 ^ (4 | rho >> 1)) << 4);
    // the (chunk, step) stages of this wave are one stream; past its end the last stage is fetched again (uniform vmcnt
    // arithmetic)
    const int64_t row0 = (int64_t)e * Nrows + c0 * CHUNK_ROWS;
    const int8_t *p0 = w0 + (row0 + (DOWN ? wave * 32 : 0)) * Kdim + s0 * 128;
    const int8_t *p1 = DOWN ? p0 : w1 + row0 * Kdim + s0 * 128;
    const unsigned second = DOWN ? 16u * (unsigned)Kdim : 0;   // of the down rows: from the first 16 to the next
    int step_left = nsw, chunk_left = nch;
    const unsigned ring_at = (unsigned)(uintptr_t)(lptr_t)ring;
    auto issue = [&](int slot) {
        const unsigned at = ring_at + slot * RX_STAGE;
        dma16(p0, woff0, at);
        dma16(p0, woff1, at + 1024);
        dma16(DOWN ? p0 : p1, woff0 + second, at + 2048);
        dma16(DOWN ? p0 : p1, woff1 + second, at + 3072);
        int by = 128;
        if (--step_left == 0) {
            step_left = nsw;
            by = CHUNK_ROWS * Kdim - (nsw - 1) * 128;
            if (--chunk_left <= 0) by = 0, step_left = 1;
        }
        p0 += by;
        if (!DOWN) p1 += by;
    };
    // weight scales (nch * SCW <= RX_SCALES) and the pair whose metadata this thread brings: requested here, parked below
    float wsc_now[4];
    if (first) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int o = min(tid + u * 256, nch * SCW - 1);
            if constexpr (DOWN) wsc_now[u] = sc0[row0 + o];
            else wsc_now[u] = ((o & 16) ? sc1 : sc0)[row0 + (o >> 5) * 16 + (o & 15)];
        }
    }
    const int pos = pos0 + min(tid, n - 1), pair = *(global_ptr<const int32_t>)(perm + pos);
    // the weight stream starts first: its addresses do not depend on the tokens, whose lookups cost two dependent memory
    // round trips
    if (nsw > 0) {
#pragma unroll
        for (int d = 0; d < RING; ++d) issue(d);
    }
    // Activation rows as MFMA fragments held in registers for every chunk: lane (token r, 16-byte chunk g_ (+4)).  Rows past
    // the segment repeat its last row and are never stored.
    const int r = lane & 15, g_ = lane >> 4;
    v4i xr[MTT][NSMAX][2];
    int last_step = steps - 1 - s0;
    asm volatile("" : "+v"(last_step));   // (scalar registers are what this kernel has fewest of)
    if constexpr (OWN) {
        // a wave a row, as the quantizer by itself, 8 or 16 rows at a time: the sums' area, which this form does not use, holds them.
        // All rows are requested before the first is used: they were written all over the chip.  (Requested one by one, 16 tokens to
        // the same eight experts took 32.9 us instead of 30.5, 92.8 -> 92.2 as a router sends them.)
        static_assert(DOWN && MTT == 1 && NSMAX * 128 <= 1024, "one pass of rows of at most two chunks a lane");
        constexpr int C = NSMAX * 128 > 512 ? 2 : 1, ROWS = 4;   // chunks a lane, rows a wave
        constexpr int AT_ONCE = RX_RED_BYTES / (NSMAX * 128) < 16 ? 8 : 16;
        static_assert(AT_ONCE * NSMAX * 128 <= RX_RED_BYTES, "");
        int8_t *const s_code = reinterpret_cast<int8_t *>(smem + RX_RING_BYTES);
        const int jq = lane & 31;
        int kd = Kdim, writes = c0;
        asm volatile("" : "+v"(kd), "+v"(writes));   // (as above)
        float v[ROWS][C][8];
        int there = n - wave;   // opaque, or the compiler keeps every comparison with it in scalar registers
#pragma unroll
        for (int k = 0; k < ROWS; ++k) {
            asm volatile("" : "+s"(there));
            const int row = 4 * k + wave;
            if (4 * k >= there) continue;
            const float *hr = h + (int64_t)(pos0 + row) * kd;
#pragma unroll
            for (int i = 0; i < C; ++i) {
                const int c = lane + 64 * i, of = (c >> 5) * 256 + 4 * jq;
                v4f lo = (v4f){0.f, 0.f, 0.f, 0.f}, hi = lo;
                if ((C == 2 && i == 0) || c * 8 < kd) {   // (two chunks a lane: rows of more than 512)
                    lo = *(global_ptr<const v4f>)(hr + of);
                    hi = *(global_ptr<const v4f>)(hr + of + 128);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) v[k][i][e] = lo[e], v[k][i][4 + e] = hi[e];
            }
        }
        static_for<16 / AT_ONCE>([&](auto Part) {
            constexpr int base = decltype(Part)::value * AT_ONCE;
            if (base >= n) return;
            if (base) __syncthreads();   // the rows before have been read
#pragma unroll
            for (int k = base / 4; k < (base + AT_ONCE) / 4; ++k) {
                asm volatile("" : "+s"(there));
                const int row = 4 * k + wave;
                if (4 * k >= there) continue;
                float amax = 0.0f;
#pragma unroll
                for (int i = 0; i < C; ++i) {
                    fwht_codes<256>(v[k][i], jq);
                    amax = fmaxf(amax, abs8(v[k][i]));
                }
                amax = max_lanes<64>(amax);
                const float sc = (amax == 0.0f) ? 1.0f : amax / 127.0f;
                const float inv = (amax == 0.0f) ? 0.0f : 127.0f / amax;
                if (lane == 0) s_tsc[row] = sc;
                if (lane == 0 && writes == 0) *(global_ptr<float>)(act_scale + pos0 + row) = sc;
                int8_t *const to = act + (int64_t)(pos0 + row) * kd;
#pragma unroll
                for (int i = 0; i < C; ++i) {
                    const int c = lane + 64 * i, of = (c >> 5) * 256 + 4 * jq;
                    if (!(C == 2 && i == 0) && c * 8 >= kd) continue;
                    const uint32_t q0 = quant4(v[k][i][0], v[k][i][1], v[k][i][2], v[k][i][3], inv), q1 = quant4(v[k][i][4], v[k][i][5], v[k][i][6], v[k][i][7], inv);
                    *reinterpret_cast<uint32_t *>(s_code + (row - base) * kd + of) = q0;
                    *reinterpret_cast<uint32_t *>(s_code + (row - base) * kd + of + 128) = q1;
                    if (writes == 0) {
                        *(global_ptr<uint32_t>)(to + of) = q0;
                        *(global_ptr<uint32_t>)(to + of + 128) = q1;
                    }
                }
            }
            __syncthreads();
            const int mine = min(r, n - 1);
            if (mine >= base && mine < base + AT_ONCE) {
                const int8_t *xp = s_code + (mine - base) * kd + g_ * 16;
#pragma unroll
                for (int i = 0; i < NSMAX; ++i) {
                    const int st = min(i, last_step) * 128;
                    xr[0][i][0] = *reinterpret_cast<const v4i *>(xp + st);
                    xr[0][i][1] = *reinterpret_cast<const v4i *>(xp + st + 64);
                }
            }
        });
    }
#pragma unroll
    for (int b = 0; b < (OWN ? 0 : MTT); ++b) {
        const int at = pos0 + min(b * 16 + r, n - 1);
        const int8_t *xp = act + (DOWN ? (int64_t)at : (int64_t)(perm[at] / topk)) * Kdim + g_ * 16 + s0 * 128;
#pragma unroll
        for (int i = 0; i < NSMAX; ++i) {
            const unsigned st = (unsigned)min(i, last_step) * 128;
            xr[b][i][0] = *reinterpret_cast<const v4i *>(xp + st);
            xr[b][i][1] = *reinterpret_cast<const v4i *>(xp + st + 64);
        }
    }
    if (tid < 16 * MTT) {
        s_dst[tid] = DOWN ? pair : pos;
        if constexpr (!OWN) s_tsc[tid] = act_scale[DOWN ? pos : pair / topk];
    }
    if (first) {
#pragma unroll
        for (int u = 0; u < 4; ++u) s_wsc[min(tid + u * 256, nch * SCW - 1)] = wsc_now[u];
    }
    __syncthreads();   // token metadata, weight scales and the zeroed sums are visible to every wave

    // read side: fragment (16-row group, K half kk): lane (row r = l%16, g_ = l/16) reads row r, chunk 4*kk + g_
    const char *frag0, *frag1;
    {
        const int rr = r & 7, par = r >> 3, sigma = (par << 2) | (rr >> 1);
        frag0 = ring + par * 1024 + ((8 * rr + (g_ ^ sigma)) << 4);
        frag1 = ring + par * 1024 + ((8 * rr + ((4 + g_) ^ sigma)) << 4);
    }
    int slot = 0;
    for (int ch = 0; ch < nch; ++ch) {
        int left = n, steps_here = nsw;   // opaque, or the compiler keeps every comparison with them in scalar registers
        asm volatile("" : "+s"(left), "+s"(steps_here));
        v4i acc[NGRP][MTT];
#pragma unroll
        for (int a = 0; a < NGRP; ++a)
#pragma unroll
            for (int b = 0; b < MTT; ++b) acc[a][b] = (v4i){0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < NSMAX; ++i) {
            asm volatile("" : "+s"(steps_here));
            if (i >= steps_here) continue;
            wait_vm<(RING - 1) * 2 * NGRP>();   // the oldest stage in flight has landed
            v4i wf[NGRP][2];
#pragma unroll
            for (int a = 0; a < NGRP; ++a) {
                wf[a][0] = *reinterpret_cast<const v4i *>(frag0 + slot * RX_STAGE + a * 2048);
                wf[a][1] = *reinterpret_cast<const v4i *>(frag1 + slot * RX_STAGE + a * 2048);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // fragments are in registers: the slot may be refilled
            issue(slot);
#pragma unroll
            for (int kk = 0; kk < 2; ++kk)
#pragma unroll
                for (int a = 0; a < NGRP; ++a)
#pragma unroll
                    for (int b = 0; b < MTT; ++b)
                        acc[a][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[a][kk], xr[b][i][kk], acc[a][b], 0, 0, 0);
            slot = slot + 1 == RING ? 0 : slot + 1;
        }
        const float *wsc = s_wsc + ch * SCW;
        // accumulator layout: lane l, register q  <->  weight row 4*(l/16)+q, token l%16
        if constexpr (!DOWN) {
            // the four K slices meet in LDS by integer atomic adds (exact, order-free); whoever reads a sum puts
            // the zero back for the next chunk
#pragma unroll
            for (int a = 0; a < NGRP; ++a)
#pragma unroll
                for (int b = 0; b < MTT; ++b)
#pragma unroll
                    for (int q = 0; q < 4; ++q) atomicAdd(&s_red[((a * MTT + b) * 4 + q) * 64 + lane], acc[a][b][q]);
            __syncthreads();
            // 16*MTT tokens x 16 channels, channel fastest; h = silu(g) * u in sorted-pair order
#pragma unroll
            for (int b = 0; b < MTT; ++b) {
                const int nl = tid & 15, row = b * 16 + (tid >> 4);
                const int bq = (b * 4 + (nl & 3)) * 64 + (nl >> 2) * 16 + (row & 15);
                const int gi = s_red[bq], ui = s_red[MTT * 256 + bq];
                s_red[bq] = 0;
                s_red[MTT * 256 + bq] = 0;
                if (row < left) {
                    const float sxt = s_tsc[row];
                    const float gv = ((float)gi * sxt) * wsc[nl];
                    const float uv = ((float)ui * sxt) * wsc[16 + nl];
                    out[(int64_t)s_dst[row] * Nrows + (c0 + ch) * 16 + nl] = silu(gv) * uv;
                }
            }
            __syncthreads();   // the zeroes are in place before the next chunk's sums arrive
        } else {
            // every wave owns its 32 rows over the whole of K: results leave straight from the accumulators, four
            // consecutive channels of one token per lane; out[pair] in pair order
#pragma unroll
            for (int a = 0; a < NGRP; ++a) {
                const int nl = wave * 32 + a * 16 + 4 * g_;
                const float4 ws = *reinterpret_cast<const float4 *>(wsc + nl);
#pragma unroll
                for (int b = 0; b < MTT; ++b) {
                    const int row = b * 16 + r;
                    if (row < left) {
                        const float ts = s_tsc[row];
                        float4 o;
                        o.x = ((float)acc[a][b][0] * ts) * ws.x;
                        o.y = ((float)acc[a][b][1] * ts) * ws.y;
                        o.z = ((float)acc[a][b][2] * ts) * ws.z;
                        o.w = ((float)acc[a][b][3] * ts) * ws.w;
                        *reinterpret_cast<float4 *>(out + (int64_t)s_dst[row] * Nrows + (c0 + ch) * 128 + nl) = o;
                    }
                }
            }
        }
    }
    wait_vm<0>();   // trailing re-fetches must not write LDS behind this pass
}

// The row chunks of all experts that have tokens, one behind the other in expert order and once per pass over them, are dealt
// evenly to two workgroups a compute unit (what LDS and registers hold): workgroup i of G takes the chunks that begin in the
// i-th of G equal shares, a run that may end one expert and begin the next.  Before, runs of a fixed length in an order by size
// filled the units twice and a bit, with half of the experts idle at 16 tokens, and every run paid its set-up.
// Bound by HBM.  Both expert kernels at H = 2048, I = 768, 128 experts, top-8, us before -> after: 16 tokens 90 -> 75,
// 512 tokens at 32 an expert 147 -> 137 (604 MB at 4.4 TB/s; 115 without the results' 46 MB of stores, 110 without the matrix
// instructions as well), 512 as a router sends them, up to 83 an expert, 156.1 -> 155.1 (gate/up 98.4 -> 96.0, down 57.7 -> 59.1:
// its shares are four or five chunks, and longer where an expert has more tokens).  The layer with a router's own counts, over 38
// shapes from 1 to 2048 tokens, 16 to 128 experts: 0.84 to 1.00 of the time before, 512 tokens 191.9 -> 186.5.  Measured without gain: non-temporal stores and loads, whole 128-byte lines per store, exact counts of
// the stores in the waits, costs that grow with an expert's tokens, rings of two stages, three workgroups a unit.
// by_chunk: at most a chunk a workgroup, all of the same cost, with the compute units' own order as the balance.
// OWN: see rx_pass.
template <bool DOWN, int NSMAX, bool OWN>
__global__ __launch_bounds__(256, 2) void k_moe_expert_rx(int8_t *act, float *act_scale, const float *__restrict__ h,
                                                          const int32_t *__restrict__ perm,
                                                          const int32_t *__restrict__ seg_off,
                                                          const int8_t *__restrict__ w0, const float *__restrict__ sc0,
                                                          const int8_t *__restrict__ w1, const float *__restrict__ sc1,
                                                          float *__restrict__ out, int Kdim, int Nrows, int topk, int chunks,
                                                          int E, int by_chunk)
{
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    constexpr int PASS = OWN ? OWN_PASS : rx_most(NSMAX);
    if constexpr (OWN) asm volatile("" : "+v"(h), "+v"(act), "+v"(act_scale), "+v"(perm));   // (scalar registers are what this kernel has fewest of)
    if constexpr (!DOWN) {
        int *s_red = reinterpret_cast<int *>(smem + RX_RING_BYTES);
        for (int o = tid; o < RX_RED_BYTES / 4; o += 256) s_red[o] = 0;
    }
    // cost of a row chunk: the passes over it (all sums fit in 31 bits: at most (65535 + 2^24 / 32) passes of 2048 chunks)
    const int per_pass = by_chunk ? INT32_MAX - (1 << 24) : PASS;
    auto cost = [&](int count) { return (int)((unsigned)(count + per_pass - 1) / (unsigned)per_pass); };
    auto segment = [&](int e, int *first, int *count) {   // of expert e, which may lie past the last one
        *first = seg_off[min(e, E)];
        *count = seg_off[min(e + 1, E)] - *first;
    };
    int total = 0;
    for (int b = 0; b < E; b += 64) {
        int s, c;
        segment(b + lane, &s, &c);
        total += __builtin_amdgcn_readlane(wave_scan(cost(c)), 63);
    }
    total *= chunks;
    const int share = total / gridDim.x, rest = total - share * gridDim.x, wg = blockIdx.x;
    const int lo = wg * share + min(wg, rest), hi = lo + share + (wg < rest ? 1 : 0);
    // the first expert that reaches past lo, and where it begins
    int e = 0, at = 0, seg0 = 0, count = 0;
    for (; e < E; e += 64) {
        int s, n;
        segment(e + lane, &s, &n);
        const int c = cost(n), incl = wave_scan(c);
        const unsigned long long past = __ballot((at + incl) * chunks > lo);
        if (past) {
            const int l = __ffsll((long long)past) - 1;
            at += __builtin_amdgcn_readlane(incl - c, l);
            seg0 = __builtin_amdgcn_readlane(s, l);
            count = __builtin_amdgcn_readlane(n, l);
            e += l;
            break;
        }
        at += __builtin_amdgcn_readlane(incl, 63);
    }
    int skip = lo - at * chunks, left = hi - at * chunks;   // of the share, from where expert e begins
    constexpr int MOST = rx_most_chunks(DOWN);   // chunks whose weight scales LDS holds
    for (; e < E && left > 0; segment(++e, &seg0, &count)) {
        const int passes = cost(count);
        const int last = passes ? min(chunks, (left + passes - 1) / passes) : 0;
        int c0 = passes ? (skip + passes - 1) / passes : 0;
        skip = 0;
        left -= passes * chunks;
        for (; c0 < last; c0 += MOST) {
            const int nch = min(MOST, last - c0);
            for (int base = 0; base < count; base += PASS) {
                const int n = min(PASS, count - base);
#define MI_RX_PASS(MT_) rx_pass<DOWN, NSMAX, MT_, OWN>(smem, act, act_scale, h, perm, w0, sc0, w1, sc1, out, Kdim, Nrows, topk, e, c0, \
                                                  nch, seg0 + base, n, base == 0)
                if (n <= 16 || PASS == 16) MI_RX_PASS(1);
                else if (n <= 32 || PASS == 32) MI_RX_PASS(PASS == 16 ? 1 : 2);
                else if (n <= 48 || PASS == 48) MI_RX_PASS(PASS <= 32 ? PASS / 16 : 3);
                else MI_RX_PASS(PASS / 16);
#undef MI_RX_PASS
            }
        }
    }
}

// y[t, n] = sum over slots in order of w[t, slot] * out[t*topk + slot, n].  A slot whose expert index lies outside
// [0, E) was never dispatched, so its row of `out` was never written: it contributes nothing.
// TOPK > 0: the slot count is known at compile time (the loads of a token are then all in flight at once); 0: any.
template <int TOPK>
__global__ __launch_bounds__(256) void k_moe_combine(const float *__restrict__ out, const float *__restrict__ w,
                                                     const int32_t *__restrict__ idx, float *__restrict__ y, int T,
                                                     int H, int topk_rt, int E)
{
    constexpr int NS = TOPK > 0 ? TOPK : MAX_TOPK;
    const int topk = TOPK > 0 ? TOPK : topk_rt;
    const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= (int64_t)T * H) return;
    const int t = (int)(i / H), n = (int)(i - (int64_t)t * H);
    // every load of the token goes out before the first use; a slot that was never dispatched is read like the
    // others (its row of the workspace exists, whatever it holds) and dropped by value
    float ws[NS];
    float4 v[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int sc = s < topk ? s : topk - 1;
        const int e = idx[(int64_t)t * topk + sc];
        const bool ok = s < topk && e >= 0 && e < E;
        ws[s] = w[(int64_t)t * topk + sc];
        v[s] = *reinterpret_cast<const float4 *>(out + ((int64_t)t * topk + sc) * H + n);
        if (!ok) { ws[s] = 0.0f; v[s] = make_float4(0.f, 0.f, 0.f, 0.f); }
    }
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        if (s < topk) {
            a.x = a.x + ws[s] * v[s].x; a.y = a.y + ws[s] * v[s].y; a.z = a.z + ws[s] * v[s].z; a.w = a.w + ws[s] * v[s].w;
        }
    }
    *reinterpret_cast<float4 *>(y + i) = a;
}

struct Layout {
    int64_t off[11];
    int64_t total;
};

static Layout layout(int64_t T, int64_t H, int64_t I, int64_t E, int64_t topk)
{
    const int64_t P = T * topk;
    const int64_t sz[11] = {T * H, T * 4, P * 4, (2 * E + 1) * 4 /* seg_off: E + 1; the rest keeps the offsets that callers know */, P * I * 4, P * I, P * 4, P * H * 4, P * 4, P * 4, T * E * 4};
    Layout L;
    int64_t o = 0;
    for (int i = 0; i < 11; ++i) { L.off[i] = o; o += align_up(sz[i], 256); }
    L.total = o;
    return L;
}

static int32_t check_shapes(int64_t T, int64_t H, int64_t I, int64_t E, int32_t topk)
{
    if (T < 0 || H <= 0 || I <= 0 || E <= 0 || topk <= 0) return MI_EINVAL;   // T == 0: an empty batch, a call that does nothing
    if (H % 128 || I % 256 || topk > MAX_TOPK || topk > E) return MI_EINVAL;
    if (H > 32768 || I > 32768 || T * topk > (1LL << 24) || E > 65535) return MI_ERANGE;
    if (2 * E * ((T + 31) / 32) + E + 1 > DISPATCH_MAX_WORDS) return MI_ERANGE;  // dispatch bitmap in LDS
    return MI_OK;
}

// can the router's first kernel also produce the FFN's activation codes? (block 128, a wave per row)
static bool route_can_quantize(int64_t H) { return H % 128 == 0 && H <= 2048; }

// logits + top-k; qx / sx non-null (and route_can_quantize(H)): the logits kernel also rotates and quantizes x;
// perm / seg non-null (and T <= ROUTE_DISPATCH_MAX_T): the top-k kernel also dispatches
static int32_t launch_route(const float *x, const float *wr, int32_t *idx, float *w, int64_t T, int64_t H, int64_t E,
                            int32_t topk, float *logits, int8_t *qx, float *sx, int32_t *perm, int32_t *seg, void *stream)
{
    // eight experts a wave (twice the workgroups) while sixteen would leave at most two workgroups to a compute unit,
    // one while eight would leave half of the units without any.  One a wave requests eight rounds of 256 floats at a time,
    // also where the row ends before: fewer token groups where that is most of them.  Router alone, us eight -> one, groups x E:
    // H = 256, 256 5.9 -> 5.3, 384 5.9 -> 6.3; H = 1024, 512 7.8 -> 6.9, 1024 7.8 -> 9.2; H = 1536, 768 9.0 -> 7.7, 1024 9.0 -> 9.4;
    // H = 3072, 1024 12.4 -> 14.0; a layer at 1024, H = 2048 67.4 -> 64.2, H = 4096 109 -> 102.
    const int64_t groups = (T + 15) / 16;
    const int cus = compute_units(), nj = (int)(H / 256);
    const int64_t few = nj == 1 ? cus / 8 : std::max(cus / 4, cus / 2 * nj / ((nj + 7) / 8 * 8));
    const int ew = groups * (E / 8) <= few ? 1 : groups * (E / 16) <= 2 * (int64_t)cus ? 8 : 16;
    // one expert a wave: a multiple of 8 in x keeps the E workgroups of a token group on one XCD, which then reads the group's
    // rows once.  It pays where the activations are more than an XCD's 4 MB of L2: router alone, 16 experts, us without -> with,
    // H = 4096, 269 tokens 11.1 -> 9.4, 1005 tokens 47.0 -> 15.6; below, the XCDs that get a group less cost more than it gives
    // (H = 2048, 64 experts, 141 tokens 7.8 -> 9.5).
    const int64_t gx = ew == 1 && T * H > (1 << 20) ? (groups + 7) / 8 * 8 : groups;
    const dim3 grid((unsigned)gx, (unsigned)(E / ew));
    const int cq = qx ? (int)((H / 8 + 63) / 64) : 0;
#define MI_LOGITS(CQ_)                                                                                                  \
    do {                                                                                                                \
        if (ew == 1)                                                                                                    \
            launch_kernel((k_moe_logits<CQ_, 1>), grid, dim3(256), 0, as_stream(stream), x, wr, logits, (int)T,    \
                          (int)H, (int)E, qx, sx);                                                                      \
        else if (ew == 8)                                                                                               \
            launch_kernel((k_moe_logits<CQ_, 8>), grid, dim3(256), 0, as_stream(stream), x, wr, logits, (int)T,    \
                          (int)H, (int)E, qx, sx);                                                                      \
        else                                                                                                            \
            launch_kernel((k_moe_logits<CQ_, 16>), grid, dim3(256), 0, as_stream(stream), x, wr, logits, (int)T,   \
                          (int)H, (int)E, qx, sx);                                                                      \
    } while (0)
    switch (cq) {
    case 0: MI_LOGITS(0); break;
    case 1: MI_LOGITS(1); break;
    case 2: MI_LOGITS(2); break;
    case 3: MI_LOGITS(3); break;
    default: MI_LOGITS(4); break;
    }
#undef MI_LOGITS
    int32_t rc = launch_status();
    if (rc) return rc;
    if (perm) {
        const size_t words = (size_t)(2 * E * ((T + 31) / 32) + E + 1);
        launch_kernel(k_moe_topk_dispatch, dim3(1), dim3(1024), words * 4, as_stream(stream), logits, idx, w, perm, seg,
                      (int)T, (int)E, (int)topk, topk_magic(topk));
        return launch_status();
    }
    launch_kernel(k_moe_topk, dim3((unsigned)((T + 3) / 4)), dim3(256), 0, as_stream(stream), logits, idx, w, (int)T,
                  (int)E, (int)topk);
    return launch_status();
}

}  // namespace moe
}  // namespace mi

using namespace mi;

extern "C" int64_t mi_moe_route_workspace_bytes(int64_t T, int64_t E)
{
    if (T < 0 || E <= 0) return MI_EINVAL;
    return moe::align_up(T * E * 4, 256);
}

extern "C" int32_t mi_moe_route(const float *x, const float *wr, int32_t *idx, float *w, int64_t T, int64_t H,
                                int64_t E, int32_t topk, void *workspace, int64_t workspace_bytes, void *stream)
{
    if (!x || !wr || !idx || !w || T < 0 || H <= 0 || E <= 0 || topk <= 0) return MI_EINVAL;
    if (H % 256 || E % 16 || topk > moe::MAX_TOPK || topk > E) return MI_EINVAL;
    if (E > 256 || T > (1LL << 24)) return MI_ERANGE;
    if (!aligned16(x) || !aligned16(wr) || !aligned4(idx) || !aligned4(w)) return MI_EINVAL;
    if (!workspace || !aligned16(workspace)) return MI_EINVAL;
    if (workspace_bytes < mi_moe_route_workspace_bytes(T, E)) return MI_ENOSPC;
    if (T == 0) return MI_OK;
    return moe::launch_route(x, wr, idx, w, T, H, E, topk, static_cast<float *>(workspace), nullptr, nullptr, nullptr,
                             nullptr, stream);
}

extern "C" int32_t mi_moe_dispatch(const int32_t *idx, int32_t *perm, int32_t *seg_off, int64_t T, int64_t E,
                                   int32_t topk, void *stream)
{
    if (!idx || !perm || !seg_off || T < 0 || E <= 0 || topk <= 0) return MI_EINVAL;
    if (T * topk > (1LL << 24) || E > 65535) return MI_ERANGE;
    const int64_t words = 2 * E * ((T + 31) / 32) + E + 1;
    if (words > moe::DISPATCH_MAX_WORDS) return MI_ERANGE;
    MI_LDS_OPT_IN((&moe::k_moe_dispatch), (int)(moe::DISPATCH_MAX_WORDS * 4));
    launch_kernel(moe::k_moe_dispatch, dim3(1), dim3(1024), (size_t)words * 4, as_stream(stream), idx, perm,
                  seg_off, (int)T, (int)E, (int)topk, moe::topk_magic(topk));
    return launch_status();
}

extern "C" int64_t mi_moe_ffn_workspace_bytes(int64_t T, int64_t H, int64_t I, int64_t E, int32_t topk)
{
    int32_t rc = moe::check_shapes(T, H, I, E, topk);
    if (rc) return rc;
    return moe::layout(T, H, I, E, topk).total;
}

extern "C" int64_t mi_moe_layer_workspace_bytes(int64_t T, int64_t H, int64_t I, int64_t E, int32_t topk)
{
    return mi_moe_ffn_workspace_bytes(T, H, I, E, topk);
}

extern "C" int64_t mi_moe_ffn_workspace_offset(int32_t which, int64_t T, int64_t H, int64_t I, int64_t E,
                                               int32_t topk)
{
    int32_t rc = moe::check_shapes(T, H, I, E, topk);
    if (rc) return rc;
    if (which < 0 || which > 10) return MI_EINVAL;
    return moe::layout(T, H, I, E, topk).off[which];
}

// codes_ready: the activation codes and scales already sit in the workspace (written by the router's first kernel)
// dispatched: so do the dispatch's outputs
static int32_t run_ffn(const float *x, const int32_t *idx, const float *w, const int8_t *wg, const float *sg,
                       const int8_t *wu, const float *su, const int8_t *wd, const float *sd, float *y, int64_t T,
                       int64_t H, int64_t I, int64_t E, int32_t topk, void *workspace, int64_t workspace_bytes,
                       void *stream, bool codes_ready, bool dispatched)
{
    int32_t rc = moe::check_shapes(T, H, I, E, topk);
    if (rc) return rc;
    if (!x || !idx || !w || !wg || !sg || !wu || !su || !wd || !sd || !y || !workspace) return MI_EINVAL;
    if (!aligned16(x) || !aligned16(wg) || !aligned16(wu) || !aligned16(wd) || !aligned16(y) || !aligned16(workspace))
        return MI_EINVAL;
    const moe::Layout L = moe::layout(T, H, I, E, topk);
    if (workspace_bytes < L.total) return MI_ENOSPC;
    if (T == 0) return MI_OK;
    char *ws = static_cast<char *>(workspace);
    int8_t *qx = reinterpret_cast<int8_t *>(ws + L.off[0]);
    float *sx = reinterpret_cast<float *>(ws + L.off[1]);
    int32_t *perm = reinterpret_cast<int32_t *>(ws + L.off[2]);
    int32_t *seg = reinterpret_cast<int32_t *>(ws + L.off[3]);
    float *h = reinterpret_cast<float *>(ws + L.off[4]);
    int8_t *hq = reinterpret_cast<int8_t *>(ws + L.off[5]);
    float *hs = reinterpret_cast<float *>(ws + L.off[6]);
    float *out = reinterpret_cast<float *>(ws + L.off[7]);
    hipStream_t s = as_stream(stream);
    const int64_t P = T * topk;

    if (!dispatched) {
        rc = mi_moe_dispatch(idx, perm, seg, T, E, topk, stream);
        if (rc) return rc;
    }
    if (!codes_ready) {
        rc = mi_fwht_quant_f32_i8(x, qx, sx, T, H, 128, stream);
        if (rc) return rc;
    }
    MI_LDS_OPT_IN((&moe::k_moe_expert_gemm<false>), moe::EXPERT_LDS);
    MI_LDS_OPT_IN((&moe::k_moe_expert_gemm<true>), moe::EXPERT_LDS);
    const int cus = compute_units();
    // Two workgroups a unit, or one per row chunk where these are fewer.  One per chunk beyond that loses where an expert needs a
    // pass or two (a layer of 512 tokens, H = 2048, I = 768, 64 experts, top-8: 158 -> 201 us), three or four a unit by 1 to 15 %.
    auto one_chunk = [&](int64_t chunks) { return (int)(chunks * std::min(E, P) <= 2 * cus); };
    const int steps_gu = (int)(H / 128), ns_gu = (steps_gu + 3) / 4;   // K steps per wave (the four waves split K)
    if (ns_gu <= 8) {
        const int chunks = (int)(I / 16), by_chunk = one_chunk(chunks);
        const dim3 grid(by_chunk ? (unsigned)(chunks * std::min<int64_t>(E, P)) : 2u * cus);
#define MI_RX_GU(NS)                                                                                            \
    do {                                                                                                        \
        MI_LDS_OPT_IN((&moe::k_moe_expert_rx<false, NS, false>), moe::RX_LDS);                                 \
        launch_kernel((moe::k_moe_expert_rx<false, NS, false>), grid, dim3(256), moe::RX_LDS, s, qx, sx,      \
                      (const float *)nullptr, perm, seg, wg, sg, wu, su, h, (int)H, (int)I, (int)topk, chunks, (int)E, by_chunk);          \
    } while (0)
        if (ns_gu <= 2) MI_RX_GU(2);
        else if (ns_gu <= 4) MI_RX_GU(4);
        else MI_RX_GU(8);
#undef MI_RX_GU
    } else {
        launch_kernel(moe::k_moe_expert_gemm<false>, dim3((unsigned)(I / 16), (unsigned)E), dim3(256),
                      moe::EXPERT_LDS, s, qx, sx, perm, seg, wg, sg, wu, su, h, (int)H, (int)I, (int)I, (int)topk,
                      1);
    }
    rc = launch_status();
    if (rc) return rc;
    const int steps_dn = (int)(I / 128);   // every wave walks the whole of K
    const bool own = steps_dn <= 8 && moe::own_codes(T, E, topk);
    if (!own) {
        rc = mi_fwht_quant_f32_i8(h, hq, hs, P, I, 256, stream);
        if (rc) return rc;
    }
    if (steps_dn <= 8) {
        const int chunks = (int)(H / 128), by_chunk = one_chunk(chunks);
        const dim3 grid(by_chunk ? (unsigned)(chunks * std::min<int64_t>(E, P)) : 2u * cus);
#define MI_RX_DN1(NS, OWN_)                                                                                     \
    do {                                                                                                        \
        MI_LDS_OPT_IN((&moe::k_moe_expert_rx<true, NS, OWN_>), moe::RX_LDS);                                    \
        launch_kernel((moe::k_moe_expert_rx<true, NS, OWN_>), grid, dim3(256), moe::RX_LDS, s, hq, hs, h, perm, seg, wd, \
                      sd, (const int8_t *)nullptr, (const float *)nullptr, out, (int)I, (int)H,                 \
                      (int)topk, chunks, (int)E, by_chunk);                                                     \
    } while (0)
#define MI_RX_DN(NS)                 \
    do {                             \
        if (own) MI_RX_DN1(NS, true); \
        else MI_RX_DN1(NS, false);   \
    } while (0)
        if (steps_dn <= 2) MI_RX_DN(2);
        else if (steps_dn <= 4) MI_RX_DN(4);
        else if (steps_dn <= 6) MI_RX_DN(6);
        else MI_RX_DN(8);
#undef MI_RX_DN
#undef MI_RX_DN1
    } else {
        launch_kernel(moe::k_moe_expert_gemm<true>, dim3((unsigned)((H + 127) / 128), (unsigned)E), dim3(256),
                      moe::EXPERT_LDS, s, hq, hs, perm, seg, wd, sd, (const int8_t *)nullptr,
                      (const float *)nullptr, out, (int)I, (int)H, (int)H, (int)topk, 1);
    }
    rc = launch_status();
    if (rc) return rc;
    const dim3 cgrid((unsigned)((T * H / 4 + 255) / 256));
#define MI_COMBINE(K_) launch_kernel(moe::k_moe_combine<K_>, cgrid, dim3(256), 0, s, out, w, idx, y, (int)T, (int)H, (int)topk, (int)E)
    switch (topk) {
    case 1: MI_COMBINE(1); break;
    case 2: MI_COMBINE(2); break;
    case 4: MI_COMBINE(4); break;
    case 8: MI_COMBINE(8); break;
    default: MI_COMBINE(0); break;
    }
#undef MI_COMBINE
    return launch_status();
}

extern "C" int32_t mi_moe_ffn(const float *x, const int32_t *idx, const float *w, const int8_t *wg, const float *sg,
                              const int8_t *wu, const float *su, const int8_t *wd, const float *sd, float *y,
                              int64_t T, int64_t H, int64_t I, int64_t E, int32_t topk, void *workspace,
                              int64_t workspace_bytes, void *stream)
{
    return run_ffn(x, idx, w, wg, sg, wu, su, wd, sd, y, T, H, I, E, topk, workspace, workspace_bytes, stream, false, false);
}

extern "C" int32_t mi_moe_layer(const float *x, const float *wr, const int8_t *wg, const float *sg, const int8_t *wu,
                                const float *su, const int8_t *wd, const float *sd, float *y, int64_t T, int64_t H,
                                int64_t I, int64_t E, int32_t topk, void *workspace, int64_t workspace_bytes,
                                void *stream)
{
    int32_t rc = moe::check_shapes(T, H, I, E, topk);
    if (rc) return rc;
    if (!workspace || !aligned16(workspace)) return MI_EINVAL;
    const moe::Layout L = moe::layout(T, H, I, E, topk);
    if (workspace_bytes < L.total) return MI_ENOSPC;
    if (T == 0) return MI_OK;
    char *ws = static_cast<char *>(workspace);
    int32_t *idx = reinterpret_cast<int32_t *>(ws + L.off[8]);
    float *w = reinterpret_cast<float *>(ws + L.off[9]);
    // the checks of mi_moe_route, which this call stands in for
    if (!x || !wr || H % 256 || E % 16 || E > 256 || !aligned16(x) || !aligned16(wr)) return MI_EINVAL;
    const bool fuse = moe::route_can_quantize(H), few = T <= moe::ROUTE_DISPATCH_MAX_T;
    rc = moe::launch_route(x, wr, idx, w, T, H, E, topk, reinterpret_cast<float *>(ws + L.off[10]),
                           fuse ? reinterpret_cast<int8_t *>(ws + L.off[0]) : nullptr,
                           fuse ? reinterpret_cast<float *>(ws + L.off[1]) : nullptr,
                           few ? reinterpret_cast<int32_t *>(ws + L.off[2]) : nullptr,
                           few ? reinterpret_cast<int32_t *>(ws + L.off[3]) : nullptr, stream);
    if (rc) return rc;
    return run_ffn(x, idx, w, wg, sg, wu, su, wd, sd, y, T, H, I, E, topk, workspace, workspace_bytes, stream, fuse, few);
}
