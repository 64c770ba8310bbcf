// W8A8 contraction for one token, and for two to four where they have few rows of a long K (decode GEMV):
//   acc[m,n] = sum_k qx[m,k] * qw[n,k],   y = ((float)acc * sx[m]) * sw[n]
// The weights [N,K] are read from HBM exactly once; everything else is small.
// Bound: HBM.  Algorithmic bytes per call = N*K (weights) + M*K (codes) + 4*M*N (output) + 4*(N+M) (scales).
//
//  k_gemv_reg: a lane always works on the same byte offsets of a weight row, so its share of the activation codes
//  lives in registers for the whole kernel: no LDS and no barrier in the streaming part, 16 x 1 KB weight loads in
//  flight per wave, v_dot4_i32_i8, one transposed butterfly per wave.
//  k_gemv_row makes the codes of its one token, or its two to four, itself (rotate + quantize, with RMSNorm or SwiGLU in front),
//  for K up to 16384 (4096).
#include <algorithm>
#include "attn_merge.h"
#include "common.h"
#include "fwht_core.h"

namespace mi {

// Transposed butterfly: `p` holds V (a power of two <= 64) per-lane partial sums; after the call lane l holds
// the wave-wide total of value  l >> (6 - log2 V)  (lanes that share those top bits hold the same total).
// Each round hands half of the values to the partner lane, so V values cost V - 1 shuffles + log-many, not 6 V.
template <int V, int OFF>
__device__ __forceinline__ void fold_sum(int (&p)[V], int lane)
{
    if constexpr (V > 1) {
        const bool hi = (lane & OFF) != 0;
        int q[V / 2];
#pragma unroll
        for (int i = 0; i < V / 2; ++i) {
            if constexpr (OFF == 32) {   // the exchange that the comment above describes is one instruction
                const auto r = __builtin_amdgcn_permlane32_swap(p[i], p[i + V / 2], false, false);
                q[i] = (int)r[0] + (int)r[1];
            } else if constexpr (OFF == 16) {
                const auto r = __builtin_amdgcn_permlane16_swap(p[i], p[i + V / 2], false, false);
                q[i] = (int)r[0] + (int)r[1];
            } else {
                const int keep = hi ? p[i + V / 2] : p[i];
                const int send = hi ? p[i] : p[i + V / 2];
                q[i] = keep + xor_lane_i<OFF>(send);
            }
        }
        fold_sum<V / 2, OFF / 2>(q, lane);
#pragma unroll
        for (int i = 0; i < V / 2; ++i) p[i] = q[i];
    } else {
        if constexpr (OFF >= 32) {
            const auto r = __builtin_amdgcn_permlane32_swap(p[0], p[0], false, false);
            p[0] = (int)r[0] + (int)r[1];
        }
        if constexpr (OFF >= 16) {
            const auto r = __builtin_amdgcn_permlane16_swap(p[0], p[0], false, false);
            p[0] = (int)r[0] + (int)r[1];
        }
        if constexpr (OFF >= 8) p[0] += xor_lane_i<8>(p[0]);
        if constexpr (OFF >= 4) p[0] += xor_lane_i<4>(p[0]);
        if constexpr (OFF >= 2) p[0] += xor_lane_i<2>(p[0]);
        if constexpr (OFF >= 1) p[0] += xor_lane_i<1>(p[0]);
    }
}

constexpr int pow2_ceil(int v) { int p = 1; while (p < v) p <<= 1; return p; }

// K = 1024 * CW * QW up to a ragged last chunk: lane l always works on the same byte offsets of a row (16*l + 1024*c
// for the wave's CW chunks).  A wave issues all the loads of its R rows at once (R*CW <= 16 x 1 KB in flight per wave),
// runs v_dot4_i32_i8 on them and reduces its R * MB per-lane sums with one transposed butterfly.  QW waves that split a row
// add their totals in LDS.  MB: tokens, M of which are there.  WG: waves of the workgroup, a multiple of QW.
template <int MB, int CW, int WG, bool DEQ>
__global__ __launch_bounds__(64 * WG) void k_gemv_reg(const int8_t *__restrict__ qx, const int8_t *__restrict__ qw,
                                                  const float *__restrict__ sx, const float *__restrict__ sw,
                                                  int32_t *__restrict__ acc_out, float *__restrict__ y, int M, int N,
                                                  int K, int QW)
{
    constexpr int R = (16 / CW) < 1 ? 1 : (16 / CW);   // rows per wave
    constexpr int V = pow2_ceil(R * MB);
    __shared__ int s_red[WG][V];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int q = wave % QW;                  // which CW-chunk slice of the row
    const int rows_per_wg = (WG / QW) * R;
    const int row0 = blockIdx.x * rows_per_wg + (wave / QW) * R;
    const int kbase = q * CW * 1024 + lane * 16;

    v4i w[R][CW];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < CW; ++c) {
            const int off = kbase + c * 1024;
            w[r][c] = (row0 + r < N && off < K) ? *reinterpret_cast<const v4i *>(qw + (int64_t)(row0 + r) * K + off)
                                                : (v4i){0, 0, 0, 0};
        }
    v4i xr[MB][CW];
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int c = 0; c < CW; ++c) {
            const int off = kbase + c * 1024, ms = MB == 1 || m < M ? m : M - 1;
            xr[m][c] = off < K ? *reinterpret_cast<const v4i *>(qx + (int64_t)ms * K + off) : (v4i){0, 0, 0, 0};
        }
    int p[V];
#pragma unroll
    for (int i = 0; i < V; ++i) p[i] = 0;
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int m = 0; m < MB; ++m) {
            int a = 0;
#pragma unroll
            for (int c = 0; c < CW; ++c) {
                a = __builtin_amdgcn_sdot4(w[r][c][0], xr[m][c][0], a, false);
                a = __builtin_amdgcn_sdot4(w[r][c][1], xr[m][c][1], a, false);
                a = __builtin_amdgcn_sdot4(w[r][c][2], xr[m][c][2], a, false);
                a = __builtin_amdgcn_sdot4(w[r][c][3], xr[m][c][3], a, false);
            }
            p[r * MB + m] = a;
        }
    fold_sum<V, 32>(p, lane);
    // lane l holds value v = l >> SH; the first lane of each group of 64/V lanes speaks for it
    constexpr int SH = 6 - __builtin_ctz(V);
    const int v = lane >> SH;
    const bool speaker = (lane & ((1 << SH) - 1)) == 0;
    int total = p[0];
    if (QW > 1) {
        if (speaker) s_red[wave][v] = total;
        __syncthreads();
        if (q == 0 && speaker) {
            for (int o = 1; o < QW; ++o) total += s_red[wave + o][v];
        }
    }
    if (q == 0 && speaker && v < R * MB) {
        const int m = v % MB, n = row0 + v / MB;
        if (n < N && m < M) {
            if constexpr (DEQ) y[(int64_t)m * N + n] = ((float)total * sx[m]) * sw[n];
            else acc_out[(int64_t)m * N + n] = total;
        }
    }
}

// k_gemv_row: the GEMV of one token with what makes its codes inside, one launch instead of two.  One workgroup of eight
// waves per compute unit (more where the rows are many); the rows of the weights are dealt evenly to the waves of the chip, and
// a wave keeps two groups of R rows in flight: the row's own loads go out first (loads return in the order they were issued),
// the first two groups right behind them (where the rows are few that is all the weights there are), and while they are on
// their way the workgroup makes the codes, with the same arithmetic as the stand-alone kernels, so that codes and scales are the
// same bits, parks them in LDS, and every lane picks up its share.  Every load is unconditional: behind a branch the compiler
// no longer counts them and waits for the weights before it touches the row.
// Bound: HBM, beside about 3 us from launch to first byte.  us, in workgroups of four waves that took 16 rows at a time and
// (K = 14336) two launches -> here: 6144 x 4096 9.4 -> 7.9, with the norm 10.7 -> 9.1; 4096 x 4096 7.2 -> 5.7; 4096 x 14336
// 19.6 -> 16.2, with SwiGLU 20.4 -> 17.8; 4096 x 2048 5.4 -> 4.1; 28672 x 4096 with the norm 22.2 -> 20.9, 131072 rows of it 89.5 ->
// 89.9.  With fewer rows than waves most of them own none and make the codes all the same: 512 x 4096 4.6 -> 3.8, 16 x 4096 4.2 ->
// 3.3, with the norm 5.2 -> 4.2, where only the workgroups that had rows were started before.
//   ROT: rotate + quantize; PLAIN: the row arrives in the rotated basis and is only quantized;
//   NORM: v = ((x (+ res)) * r) * g with r = 1 / sqrt(mean((x + res)^2) + eps), then rotate + quantize; workgroup 0 also leaves
//   the residual sum (h_out) and, on request, the normalized row (xn_out);
//   SWIGLU: v = silu(gate) * up of a row [gate | up], then rotate + quantize; workgroup 0 leaves v in xn_out on request.
//   MERGED: the row of one token's attention, merged here from the partial results of up to MERGED_MOST splits (x, and their maxima
//   and sums in g), then quantized as it is.  A merge of its own is a launch of 2.4 us whose 16 KB every workgroup then reads; here
//   each reads the splits' rows, 98 KB for six, and workgroup 0 leaves the merged row in xn_out.  us of attention and projection of one sequence in a chain of
//   them, 8 kv heads, 4096 -> 4096: 1531 tokens (6 splits) 11.9 -> 10.3, 2048 (8) 12.2 -> 10.9; 4 kv heads, 2048 -> 2048, 2048 tokens 9.5 -> 8.9.
// Workgroup 0 leaves codes and scale for the caller.
enum RowOp { ROT, PLAIN, NORM, SWIGLU, MERGED };
constexpr int MERGED_MOST = 8;
struct RowArgs {
    const float *res, *g;
    float *h_out, *xn_out;
    float eps;
    int splits, group;   // MERGED: splits, query heads a kv head
};

// CW: 1024-byte chunks of a weight row, the last one shorter unless WHOLE.  MB: tokens, M of which are there (the last one is made
// again for the others), each with a row of its own at K floats from the one before.
template <int CW, bool WHOLE, int R, RowOp OP, int MB>
__global__ __launch_bounds__(512, 2) void k_gemv_row(const float *__restrict__ x, const int8_t *__restrict__ qw,
                                                     const float *__restrict__ sw, float *__restrict__ y,
                                                     int8_t *__restrict__ qx_out, float *__restrict__ sx_out, int N, int K, int M,
                                                     RowArgs ra)
{
    static_assert(MB == 1 || MB == 2 || MB == 4, "");
    static_assert(MB == 1 || OP == ROT || OP == NORM, "");
    constexpr int BLOCK = 128, LPB = BLOCK / 8, WG = 8;
    constexpr int V = pow2_ceil(R * MB), CQ = (CW + 3) / 4;   // chunks of 8 floats a thread
    __shared__ __attribute__((aligned(16))) int8_t s_x[MB][CW * 1024];   // codes
    __shared__ float s_max[MB][WG], s_sum[MB][WG * CQ];                  // row maxima, sums of squares
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned waves = gridDim.x * WG, id = blockIdx.x * WG + wave;
    // Where two groups a wave do not cover the rows, they are dealt in rounds, a group to a wave, so that the chip reads one
    // stretch of the weights at a time.  With a stretch of its own for every wave (as where two groups do) some 4096 streams run a
    // fixed distance apart, and meet in the same channels where that is near a power of two.  us, stretches -> rounds: 131072 x 2048
    // 58.9 -> 44.0, 65536 x 2048 24.6 -> 20.8, 98304 x 4096 79.8 -> 67.8, 131072 x 4096 with the norm 104.6 -> 89.9, 28672 x 4096
    // 21.3 -> 20.7.
    const bool rounds = N > 2 * R * waves;
    const int next = rounds ? R * waves : R;   // from a group of rows to the wave's next
    const int row0 = rounds ? R * id : (int)((unsigned)N * id / waves), row1 = rounds ? N : (int)((unsigned)N * (id + 1) / waves);
    const int kbase = lane * 16;
    // (no branch around a load: the compiler would wait for all of them where it cannot count them.  Past the wave's rows one
    // of them is fetched again, past a row's end its last 16 bytes)
    const int klast = WHOLE ? (CW - 1) * 1024 : min((CW - 1) * 1024, K - 16 - kbase);
    auto load_w = [&](v4i (&w)[R][CW], int row) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int8_t *const p = qw + (int64_t)min(row + r, max(row1 - 1, 0)) * K + kbase;
#pragma unroll
            for (int c = 0; c < CW; ++c) w[r][c] = *reinterpret_cast<const v4i *>(p + (c + 1 < CW ? c * 1024 : klast));
        }
    };

    // thread t owns chunks t, t + 512, ... of the row, in the layout of fwht_core.h
    const int j = tid % LPB, nchunk = K / 8;
    const bool keeper = blockIdx.x == 0;
    float v[MB][CQ][8];
    int base[CQ];
    float4 gl[CQ], gh[CQ], rl[MB][CQ], rh[MB][CQ];
    attn::Partials<OP == MERGED ? MERGED_MOST : 1, false> part;
    static_assert(OP != MERGED || CQ == 1, "a head's chunk a thread");
#pragma unroll
    for (int i = 0; i < CQ; ++i) {
        const int c = tid + i * 512;
        base[i] = (c / LPB) * BLOCK + 4 * j;
        if (OP == MERGED) {
            const int head = min(c, nchunk - 1) / LPB, kv = head / ra.group, hl = head - kv * ra.group;
            part.load(ra.g + kv * ra.splits * 8, x + ((int64_t)kv * ra.splits * 4 + hl) * BLOCK, ra.splits, hl, j);
        } else if (c < nchunk) {
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                const int64_t of = MB == 1 ? base[i] : (int64_t)min(m, M - 1) * K + base[i];
                const float4 lo = *reinterpret_cast<const float4 *>(x + of);
                const float4 hi = *reinterpret_cast<const float4 *>(x + of + BLOCK / 2);
                v[m][i][0] = lo.x; v[m][i][1] = lo.y; v[m][i][2] = lo.z; v[m][i][3] = lo.w;
                v[m][i][4] = hi.x; v[m][i][5] = hi.y; v[m][i][6] = hi.z; v[m][i][7] = hi.w;
                if constexpr (OP == NORM) {
                    if (ra.res) {
                        rl[m][i] = *reinterpret_cast<const float4 *>(ra.res + of);
                        rh[m][i] = *reinterpret_cast<const float4 *>(ra.res + of + BLOCK / 2);
                    }
                }
            }
            if constexpr (OP == NORM) {
                gl[i] = *reinterpret_cast<const float4 *>(ra.g + base[i]);
                gh[i] = *reinterpret_cast<const float4 *>(ra.g + base[i] + BLOCK / 2);
            }
            if constexpr (OP == SWIGLU) {
                gl[i] = *reinterpret_cast<const float4 *>(x + K + base[i]);
                gh[i] = *reinterpret_cast<const float4 *>(x + K + base[i] + BLOCK / 2);
            }
        } else {
#pragma unroll
            for (int m = 0; m < MB; ++m)
#pragma unroll
                for (int e = 0; e < 8; ++e) v[m][i][e] = 0.0f;
        }
    }
    v4i wa[R][CW], wb[R][CW];
    load_w(wa, row0);
    load_w(wb, row0 + next);

    auto leave = [&](float *to) {   // the rows as they stand
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
            for (int i = 0; i < CQ; ++i)
                if (tid + i * 512 < nchunk && (MB == 1 || m < M)) {
                    float *const at = to + (int64_t)m * K + base[i];
                    *reinterpret_cast<float4 *>(at) = make_float4(v[m][i][0], v[m][i][1], v[m][i][2], v[m][i][3]);
                    *reinterpret_cast<float4 *>(at + BLOCK / 2) = make_float4(v[m][i][4], v[m][i][5], v[m][i][6], v[m][i][7]);
                }
    };
    if constexpr (OP == NORM) {
        float ss[MB][CQ];   // per chunk, then per group of 64 chunks (group wave + 8 i): the order of fwht_core.h
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
            for (int i = 0; i < CQ; ++i) {
                float (&w)[8] = v[m][i];
                ss[m][i] = 0.0f;
                if (tid + i * 512 < nchunk) {
                    if (ra.res) {
                        const float4 &lo = rl[m][i], &hi = rh[m][i];
                        w[0] = w[0] + lo.x; w[1] = w[1] + lo.y; w[2] = w[2] + lo.z; w[3] = w[3] + lo.w;
                        w[4] = w[4] + hi.x; w[5] = w[5] + hi.y; w[6] = w[6] + hi.z; w[7] = w[7] + hi.w;
                    }
                    ss[m][i] = chunk_sumsq(w);
                }
            }
        if (ra.res && keeper) leave(ra.h_out);
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
            for (int i = 0; i < CQ; ++i) {
                ss[m][i] = group_sum(ss[m][i]);
                if (lane == 0) s_sum[m][wave + WG * i] = ss[m][i];
            }
        __syncthreads();
#pragma unroll
        for (int m = 0; m < MB; ++m) {
            const float total = tree_sum<WG * CQ>(s_sum[m]);
            const float r = 1.0f / sqrtf(total / (float)K + ra.eps);
#pragma unroll
            for (int i = 0; i < CQ; ++i)
                if (tid + i * 512 < nchunk) {
                    float (&w)[8] = v[m][i];
                    w[0] = (w[0] * r) * gl[i].x; w[1] = (w[1] * r) * gl[i].y;
                    w[2] = (w[2] * r) * gl[i].z; w[3] = (w[3] * r) * gl[i].w;
                    w[4] = (w[4] * r) * gh[i].x; w[5] = (w[5] * r) * gh[i].y;
                    w[6] = (w[6] * r) * gh[i].z; w[7] = (w[7] * r) * gh[i].w;
                }
        }
    }
    if constexpr (OP == SWIGLU) {
#pragma unroll
        for (int i = 0; i < CQ; ++i) {
            const float up[8] = {gl[i].x, gl[i].y, gl[i].z, gl[i].w, gh[i].x, gh[i].y, gh[i].z, gh[i].w};
            if (tid + i * 512 < nchunk) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[0][i][e] = silu(v[0][i][e]) * up[e];
            }
        }
    }
    if constexpr (OP == MERGED) {
        float l = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[0][0][e] = 0.0f;
        part.add(ra.splits, v[0][0], l);
        attn::normalize_row(l, v[0][0]);
        if (tid >= nchunk)
#pragma unroll
            for (int e = 0; e < 8; ++e) v[0][0][e] = 0.0f;
    }
    if constexpr (OP == NORM || OP == SWIGLU || OP == MERGED) {
        if (keeper && ra.xn_out) leave(ra.xn_out);
    }
#pragma unroll
    for (int m = 0; m < MB; ++m) {
        float amax = 0.0f;
#pragma unroll
        for (int i = 0; i < CQ; ++i) {
            if constexpr (OP != PLAIN && OP != MERGED) fwht_codes<BLOCK>(v[m][i], j);
            amax = fmaxf(amax, abs8(v[m][i]));
        }
        amax = max_lanes<64>(amax);
        if (lane == 0) s_max[m][wave] = amax;
    }
    __syncthreads();
    float scs[MB];
#pragma unroll
    for (int m = 0; m < MB; ++m) {
        float a = s_max[m][0];
#pragma unroll
        for (int w = 1; w < WG; ++w) a = fmaxf(a, s_max[m][w]);
        const float sc = (a == 0.0f) ? 1.0f : a / 127.0f;
        const float inv = (a == 0.0f) ? 0.0f : 127.0f / a;
        scs[m] = sc;
        if (MB > 1 && m >= M) continue;
        if (keeper && tid == 0) sx_out[m] = sc;
#pragma unroll
        for (int i = 0; i < CQ; ++i)
            if (tid + i * 512 < nchunk) {
                const uint32_t c0 = quant4(v[m][i][0], v[m][i][1], v[m][i][2], v[m][i][3], inv);
                const uint32_t c1 = quant4(v[m][i][4], v[m][i][5], v[m][i][6], v[m][i][7], inv);
                *reinterpret_cast<uint32_t *>(s_x[m] + base[i]) = c0;
                *reinterpret_cast<uint32_t *>(s_x[m] + base[i] + BLOCK / 2) = c1;
                if (keeper) {
                    int8_t *const to = qx_out + (int64_t)m * K + base[i];
                    *reinterpret_cast<uint32_t *>(to) = c0;
                    *reinterpret_cast<uint32_t *>(to + BLOCK / 2) = c1;
                }
            }
    }
    __syncthreads();

    v4i xr[MB][CW];
#pragma unroll
    for (int m = 0; m < MB; ++m) {
        const int8_t *const from = s_x[MB == 1 ? 0 : min(m, M - 1)] + kbase;
#pragma unroll
        for (int c = 0; c < CW; ++c) xr[m][c] = *reinterpret_cast<const v4i *>(from + c * 1024);
        if (!WHOLE && kbase + (CW - 1) * 1024 >= K) xr[m][CW - 1] = (v4i){0, 0, 0, 0};
    }
    // value r * MB + m of a group: row r of token m
    constexpr int SH = 6 - __builtin_ctz(V);
    const int vi = lane >> SH, mi = vi % MB, ri = vi / MB;
    const bool speaker = (lane & ((1 << SH) - 1)) == 0 && ri < R && (MB == 1 || mi < M);
    float sc = scs[0];
#pragma unroll
    for (int m = 1; m < MB; ++m) sc = mi == m ? scs[m] : sc;
    float *const yt = y + (int64_t)mi * N + ri;
    auto rows = [&](v4i (&w)[R][CW], int row) {
        int p[V];
#pragma unroll
        for (int i = 0; i < V; ++i) p[i] = 0;
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                int d = 0;
#pragma unroll
                for (int c = 0; c < CW; ++c)
#pragma unroll
                    for (int q = 0; q < 4; ++q) d = __builtin_amdgcn_sdot4(w[r][c][q], xr[m][c][q], d, false);
                p[r * MB + m] = d;
            }
        fold_sum<V, 32>(p, lane);
        if (speaker && row + ri < row1) yt[row] = ((float)p[0] * sc) * sw[row + ri];
    };
    int row = row0;
#pragma unroll 1
    for (; row + 2 * next < row1; row += 2 * next) {
        rows(wa, row);
        load_w(wa, row + 2 * next);
        rows(wb, row + next);
        load_w(wb, row + 3 * next < row1 ? row + 3 * next : row + 2 * next);
    }
    rows(wa, row);
    if (row + next < row1) rows(wb, row + next);
}

// The split of the rows by their number a wave, as far as registers go (two groups of R rows of CW chunks).  Few rows: one
// workgroup a unit whose two groups cover them.  Many: two a unit with a row at a time (20000 x 4096 and the norm 18.0 us, one a
// unit with four rows at a time 19.9), three where the codes are quickly made or the rows many enough not to mind (28672 x 4096 24.9
// against 25.9 us; with the norm 21.4 against 20.4, of 65536 rows 44.9 against 45.9).  From five chunks on two a unit pay beyond six
// rows a wave only (16384 x 5120 and the norm 18.2 -> 16.1, 6144 x 8192 12.9 -> 13.9), above eight chunks one is what the registers
// hold.
template <int CW, bool WHOLE, RowOp OP, int MB>
static void start_row(int cus, int per_wave, const float *x, const int8_t *qw, const float *sw, float *y, int8_t *qx, float *sx,
                      int N, int K, int M, const RowArgs &ra, hipStream_t s)
{
    auto go = [&](auto R, int wgs) {
        launch_kernel((k_gemv_row<CW, WHOLE, decltype(R)::value, OP, MB>), dim3((unsigned)(wgs * cus)), dim3(512), 0, s, x, qw, sw,
                      y, qx, sx, N, K, M, ra);
    };
    using std::integral_constant;
    if constexpr (OP == MERGED) {   // one workgroup a unit, see merged_takes
        if (per_wave <= 2) go(integral_constant<int, 1>{}, 1);
        else if (CW > 2 || per_wave <= 4) go(integral_constant<int, 2>{}, 1);
        else if constexpr (CW <= 2) go(integral_constant<int, 4>{}, 1);
    } else if constexpr (MB == 4) {   // many rows, see rows_take
        go(integral_constant<int, 1>{}, 2);
    } else {
        if (per_wave <= 2) return go(integral_constant<int, 1>{}, 1);
        if constexpr (CW <= 4) {
            if (per_wave <= 4) return go(integral_constant<int, 2>{}, 1);
            if constexpr (CW <= 2)
                if (per_wave <= 8) return go(integral_constant<int, 4>{}, 1);
            return go(integral_constant<int, 1>{}, MB == 1 && CW == 4 && per_wave > (OP == NORM ? 20 : 10) ? 3 : 2);
        }
        go(integral_constant<int, 1>{}, CW <= 8 && per_wave > 6 ? 2 : 1);
    }
}

// Where the one kernel is the faster form, against making the codes and contracting them one behind the other: linear, norm and
// SwiGLU, 20 K from 128 to 16384, whole chunks and not, 16 to 131072 rows, weights from HBM.  Up to eight rows a wave 0.57 to 1.04
// of their time (6144 x 5120 11.9 -> 8.7 us, 4096 x 12288 with the norm 17.1 -> 14.6; no gain for 16 rows of 16384).  Up to twenty
// 0.77 to 1.00 from K = 1024 to 8192; shorter rows lose the time that a row costs beside its bytes (28672 x 640 8.3 -> 8.5), longer
// ones stream no better than in the GEMV by itself (28672 x 14336 72.6 -> 74.0 with SwiGLU).  Beyond, 0.93 to 0.97 in two to four
// whole chunks (131072 x 2048 49.4 -> 44.0), up to 1.14 elsewhere.
bool row_takes(int64_t N, int64_t K)
{
    const int64_t cus = compute_units();
    return K % 128 == 0 && K <= 16384 &&
           (N <= 64 * cus || (K >= 1024 && K <= 8192 && N <= 160 * cus) || (K >= 2048 && K <= 4096 && K % 1024 == 0));
}

// Every workgroup reads every split: up to MERGED_MOST of them and 4096 values (128 KB).  So as long as the rows go to one workgroup
// a unit: attention and projection 0.92 to 0.99 of the time with a merge of its own (1024 to 4096 values, three to eight splits, 1024
// to 16384 rows).  With two or three a unit 0.96 to 1.03 (2048 tokens, 12304 x 4096 17.9 -> 18.4, 28672 x 4096 27.9 -> 28.6, 768 tokens,
// 20480 x 1024 14.2 -> 14.4).
bool merged_takes(int splits, int64_t N, int64_t K)
{
    return splits > 1 && splits <= MERGED_MOST && K >= 1024 && K <= 4096 && row_takes(N, K) &&
           N <= (K <= 2048 ? 64 : 32) * (int64_t)compute_units();
}

template <RowOp OP>
static int32_t launch_row(const float *x, const int8_t *qw, const float *sw, float *y, int8_t *qx, float *sx, int64_t N,
                          int64_t K, const RowArgs &ra, hipStream_t s)
{
    // Every workgroup reads the whole row while others write, so buffers that share memory get the launches one behind the
    // other.  (The weights are not looked at: results on top of them are no more defined in the contraction alone.)
    if (!row_takes(N, K) || !apart({{x, (OP == SWIGLU ? 2 : 1) * K * 4}, {ra.res, K * 4}, {ra.g, K * 4}},
                                   {{y, N * 4}, {qx, K}, {sx, 4}, {ra.h_out, K * 4}, {ra.xn_out, K * 4}}))
        return MI_EINVAL;
    const int cus = compute_units(), per_wave = (int)((N + 8 * cus - 1) / (8 * cus));
    switch ((K + 1023) >> 10) {
#define MI_ROW(CW_)                                                                                                          \
    case CW_:                                                                                                                \
        if (K % 1024) start_row<CW_, false, OP, 1>(cus, per_wave, x, qw, sw, y, qx, sx, (int)N, (int)K, 1, ra, s);            \
        else start_row<CW_, true, OP, 1>(cus, per_wave, x, qw, sw, y, qx, sx, (int)N, (int)K, 1, ra, s);                      \
        break;
        MI_ROW(1) MI_ROW(2) MI_ROW(3) MI_ROW(4) MI_ROW(5) MI_ROW(6) MI_ROW(7) MI_ROW(8)
    default:
        if constexpr (OP != PLAIN)   // (an attention row has at most 64 heads)
            switch ((K + 1023) >> 10) {
                MI_ROW(9) MI_ROW(10) MI_ROW(11) MI_ROW(12) MI_ROW(13) MI_ROW(14) MI_ROW(15) MI_ROW(16)
#undef MI_ROW
            }
        else return MI_EINVAL;
    }
    return launch_status();
}

// The same for two tokens, and for three and four where the rows are many: every workgroup makes all the codes, which two launches
// do once.  us of two launches -> one, weights from HBM, linear and with the norm, K = 512 to 4096, N = 16 to 40960: two tokens 0.69 to
// 1.00 of the time and 0.77 to 0.97 (4096 x 4096 7.6 -> 5.7 and 7.7 -> 6.7, 28672 x 4096 25.3 -> 21.3 and 24.0 -> 20.8).  Three and four
// from 80 rows a unit on: linear from K = 2048 on 0.85 to 1.00 (four, 28672 x 4096 25.7 -> 22.4), fewer and shorter rows 0.87 to 1.11;
// with the norm, whose prologue is the longer, at K = 4096 0.87 to 1.02 (four, 28672 x 4096 23.8 -> 22.3, 22000 x 4096 21.2 -> 19.4,
// at worst 20496 x 4096 and a residual 19.0 -> 19.4), 0.95 to 1.18 below it (20496 x 2048 11.6 -> 12.9, 24576 x 3072 17.4 -> 18.2,
// 24576 x 3456 18.4 -> 20.0, 40960 x 2048 19.4 -> 18.6).
static bool rows_take(int64_t M, int64_t N, int64_t K, bool norm)
{
    if (M < 2 || M > 4 || K > 4096 || !row_takes(N, K)) return false;
    return M == 2 || (K >= (norm ? 4096 : 2048) && N > 80 * compute_units());
}

template <RowOp OP>
static int32_t launch_rows_of(const float *x, const int8_t *qw, const float *sw, float *y, int8_t *qx, float *sx, int64_t M,
                              int64_t N, int64_t K, const RowArgs &ra, hipStream_t s)
{
    if (!rows_take(M, N, K, OP == NORM) || !apart({{x, M * K * 4}, {ra.res, M * K * 4}, {ra.g, K * 4}},
                                      {{y, M * N * 4}, {qx, M * K}, {sx, M * 4}, {ra.h_out, M * K * 4}, {ra.xn_out, M * K * 4}}))
        return MI_EINVAL;
    const int cus = compute_units(), per_wave = (int)((N + 8 * cus - 1) / (8 * cus));
    switch ((K + 1023) >> 10) {
#define MI_ROWS1(CW_, WHOLE_, MB_) start_row<CW_, WHOLE_, OP, MB_>(cus, per_wave, x, qw, sw, y, qx, sx, (int)N, (int)K, (int)M, ra, s)
    // (three and four with the norm: four whole chunks)
#define MI_ROWS(CW_)                                                          \
    case CW_:                                                                 \
        if (M == 2 && K % 1024) MI_ROWS1(CW_, false, 2);                      \
        else if (M == 2) MI_ROWS1(CW_, true, 2);                              \
        else if constexpr (CW_ < (OP == NORM ? 4 : 2)) return MI_EINVAL;      \
        else if (OP != NORM && K % 1024) MI_ROWS1(CW_, OP == NORM, 4);        \
        else MI_ROWS1(CW_, true, 4);                                          \
        break;
        MI_ROWS(1) MI_ROWS(2) MI_ROWS(3) MI_ROWS(4)
#undef MI_ROWS
#undef MI_ROWS1
    default: return MI_EINVAL;
    }
    return launch_status();
}

int32_t launch_linear_fused(const float *x, const int8_t *qw, const float *sw, float *y, int8_t *qx, float *sx,
                            int64_t M, int64_t N, int64_t K, hipStream_t s, bool rotate)
{
    const RowArgs none = {};
    if (M != 1) return rotate ? launch_rows_of<ROT>(x, qw, sw, y, qx, sx, M, N, K, none, s) : MI_EINVAL;
    return rotate ? launch_row<ROT>(x, qw, sw, y, qx, sx, N, K, none, s) : launch_row<PLAIN>(x, qw, sw, y, qx, sx, N, K, none, s);
}

// The projection of one token's attention row from its partial results (the layout of attn_merge.h), row, codes and scale left for
// the caller: part_o and part_ml are not touched by the outputs.  MI_EINVAL: not covered, merge first.
int32_t launch_merged_linear(const float *part_o, const float *part_ml, int splits, int group, const int8_t *qw, const float *sw,
                             float *y, float *row, int8_t *qx, float *sx, int64_t N, int64_t K, hipStream_t s)
{
    if (!merged_takes(splits, N, K)) return MI_EINVAL;
    RowArgs ra = {};
    ra.g = part_ml;
    ra.xn_out = row;
    ra.splits = splits;
    ra.group = group;
    const int cus = compute_units(), per_wave = (int)((N + 8 * cus - 1) / (8 * cus));
    switch ((K + 1023) >> 10) {
#define MI_MERGED(CW_)                                                                                                              \
    case CW_:                                                                                                                       \
        if (CW_ > 1 && K % 1024) start_row<CW_, CW_ == 1, MERGED, 1>(cus, per_wave, part_o, qw, sw, y, qx, sx, (int)N, (int)K, 1, ra, s); \
        else start_row<CW_, true, MERGED, 1>(cus, per_wave, part_o, qw, sw, y, qx, sx, (int)N, (int)K, 1, ra, s);                    \
        break;
        MI_MERGED(1) MI_MERGED(2) MI_MERGED(3) MI_MERGED(4)
#undef MI_MERGED
    default: return MI_EINVAL;
    }
    return launch_status();
}

// the same with the (residual +) RMSNorm, or SwiGLU of a row [gate | up], in front
int32_t launch_norm_linear_fused(const float *x, const float *res, const float *g, float eps, float *h_out,
                                 float *xn_out, const int8_t *qw, const float *sw, float *y, int8_t *qx, float *sx,
                                 int64_t M, int64_t N, int64_t K, hipStream_t s)
{
    const RowArgs ra{res, g, h_out, xn_out, eps};
    return M == 1 ? launch_row<NORM>(x, qw, sw, y, qx, sx, N, K, ra, s) : launch_rows_of<NORM>(x, qw, sw, y, qx, sx, M, N, K, ra, s);
}
int32_t launch_swiglu_linear_fused(const float *gate_up, float *h_out, const int8_t *qw, const float *sw, float *y, int8_t *q,
                                   float *scale, int64_t M, int64_t N, int64_t K, hipStream_t s)
{
    if (M != 1) return MI_EINVAL;
    return launch_row<SWIGLU>(gate_up, qw, sw, y, q, scale, N, K, RowArgs{nullptr, nullptr, nullptr, h_out, 0.0f}, s);
}

template <int MB, int CW, int WG, bool DEQ>
static int32_t launch_reg(const int8_t *qx, const float *sx, const int8_t *qw, const float *sw, int32_t *acc,
                          float *y, int M, int N, int K, int QW, hipStream_t s)
{
    constexpr int R = (16 / CW) < 1 ? 1 : (16 / CW);
    const int rows_per_wg = (WG / QW) * R;
    const unsigned grid = (unsigned)((N + rows_per_wg - 1) / rows_per_wg);
    launch_kernel((k_gemv_reg<MB, CW, WG, DEQ>), dim3(grid), dim3(64 * WG), 0, s, qx, qw, sx, sw, acc, y, M, N, K, QW);
    return launch_status();
}

// Waves that share a row: the fewest whose shares of K = 1024 * chunks are equal and at most 7 chunks, else the fewest
// whose shares are at most 7 chunks (the last wave's is shorter); 0: more than 16.
static int gemv_split(int K)
{
    const int nchunk = (K + 1023) >> 10;
    for (int QW = 1; QW <= 4; QW <<= 1)
        if (nchunk % QW == 0 && nchunk / QW <= 7) return QW;
    for (int QW = 2; QW <= 16; QW <<= 1)
        if (nchunk <= 7 * QW) return QW;
    return 0;
}

// Whether the GEMV takes M tokens, by measurement against the small-tile kernel (weights from HBM, us GEMV : small tiles).
// One token: wherever K splits (11264 -> 1024 4.9 : 7.9, 15360 -> 256 4.2 : 9.2, 27648 -> 28672 123.5 : 133), but for shares so
// uneven that the waves move more than a tenth less than they could (9, 17 or 33 chunks): there from 12 to 40 rows a unit are
// faster in small tiles (8320 -> 8192 14.0 : 13.3, 33792 -> 4096 22.9 : 21.9), fewer and more are not (8320 -> 2048 6.5 : 7.5,
// 17408 -> 14336 43.1 : 44.4).
// Two to four: the small tiles read the codes once per 16 rows instead of once per one to three rows and win (2 tokens,
// 2048 -> 1024 2.8 : 2.5), but up to 8 rows a unit they leave half of the units idle behind a long chain of stages:
// 2 tokens, 5632 -> 512 3.6 : 4.3, 7168 -> 1024 4.1 : 4.7, 8064 -> 2048 6.1 : 7.1, and 4 tokens, 7168 -> 512 4.4 : 4.6,
// 8064 -> 2048 6.7 : 6.9.  The lines lie where the two met in a scan of K from 2048 to 7808 in steps of 384 and N from 16 to
// 3072, for each number of tokens.
bool gemv_takes(int M, int N, int K, int cus)
{
    const int QW = gemv_split(K), nchunk = (K + 1023) >> 10;
    if (!QW) return false;
    if (M == 1) return 10 * QW * ((nchunk + QW - 1) / QW) <= 11 * nchunk || N <= 12 * cus || N > 40 * cus;
    if (M > 4 || K >= 8192) return false;
    return M == 2 ? (N <= 5 * cus && K > 3072) || (N <= 8 * cus && K > 4096) || (N <= 12 * cus && K > 7168)
                  : (N <= 6 * cus && K > 5120) || (N <= 8 * cus && K > 5760);
}

template <int MB, int CW0, int WG, bool DEQ>
static int32_t launch_tokens(const int8_t *qx, const float *sx, const int8_t *qw, const float *sw, int32_t *acc, float *y,
                             int M, int N, int K, int QW, hipStream_t s)
{
    switch ((((K + 1023) >> 10) + QW - 1) / QW) {
    case 1: if constexpr (CW0 <= 1) return launch_reg<MB, 1, WG, DEQ>(qx, sx, qw, sw, acc, y, M, N, K, QW, s); break;
    case 2: if constexpr (CW0 <= 2) return launch_reg<MB, 2, WG, DEQ>(qx, sx, qw, sw, acc, y, M, N, K, QW, s); break;
    case 3: if constexpr (CW0 <= 3) return launch_reg<MB, 3, WG, DEQ>(qx, sx, qw, sw, acc, y, M, N, K, QW, s); break;
    case 4: return launch_reg<MB, 4, WG, DEQ>(qx, sx, qw, sw, acc, y, M, N, K, QW, s);
    case 5: return launch_reg<MB, 5, WG, DEQ>(qx, sx, qw, sw, acc, y, M, N, K, QW, s);
    case 6: return launch_reg<MB, 6, WG, DEQ>(qx, sx, qw, sw, acc, y, M, N, K, QW, s);
    case 7: return launch_reg<MB, 7, WG, DEQ>(qx, sx, qw, sw, acc, y, M, N, K, QW, s);
    }
    return MI_EINVAL;
}

// for what gemv_takes
template <bool DEQ>
int32_t launch_gemv(const int8_t *qx, const float *sx, const int8_t *qw, const float *sw, int32_t *acc, float *y,
                    int64_t M64, int64_t N64, int64_t K64, hipStream_t s)
{
    const int M = (int)M64, N = (int)N64, K = (int)K64;
    const int QW = gemv_split(K);
    if (M < 1 || M > 4 || !QW || (M > 1 && QW > 2)) return MI_EINVAL;
    if (QW == 16) return launch_tokens<1, 4, 16, DEQ>(qx, sx, qw, sw, acc, y, M, N, K, QW, s);   // 57 to 112 chunks
    if (QW == 8) return launch_tokens<1, 4, 8, DEQ>(qx, sx, qw, sw, acc, y, M, N, K, QW, s);     // 29 to 56
    if (M == 1) return launch_tokens<1, 1, 4, DEQ>(qx, sx, qw, sw, acc, y, M, N, K, QW, s);
    if (M == 2) return launch_tokens<2, 4, 4, DEQ>(qx, sx, qw, sw, acc, y, M, N, K, QW, s);      // four to eight
    return launch_tokens<4, 4, 4, DEQ>(qx, sx, qw, sw, acc, y, M, N, K, QW, s);
}

template int32_t launch_gemv<true>(const int8_t *, const float *, const int8_t *, const float *, int32_t *, float *,
                                   int64_t, int64_t, int64_t, hipStream_t);
template int32_t launch_gemv<false>(const int8_t *, const float *, const int8_t *, const float *, int32_t *, float *,
                                    int64_t, int64_t, int64_t, hipStream_t);

}  // namespace mi
