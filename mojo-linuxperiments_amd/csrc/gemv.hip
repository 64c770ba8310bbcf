// W8A8 contraction for one token, and for two to four where they have few rows of a long K (decode GEMV):
//   acc[m,n] = sum_k qx[m,k] * qw[n,k],   y = ((float)acc * sx[m]) * sw[n]
// The weights [N,K] are read from HBM exactly once; everything else is small.
// Bound: HBM.  Algorithmic bytes per call = N*K (weights) + M*K (codes) + 4*M*N (output) + 4*(N+M) (scales).
//
//  k_gemv_reg: a lane always works on the same byte offsets of a weight row, so its share of the activation codes
//  lives in registers for the whole kernel: no LDS and no barrier in the streaming part, 16 x 1 KB weight loads in
//  flight per wave, v_dot4_i32_i8, one transposed butterfly per wave.
//  k_gemv_fused is the same kernel with the rotate + quantize prologue (and optionally the RMSNorm) inside, for
//  one token and K <= 4096.
#include <algorithm>
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
            const int keep = hi ? p[i + V / 2] : p[i];
            const int send = hi ? p[i] : p[i + V / 2];
            q[i] = keep + __shfl_xor(send, OFF, 64);
        }
        fold_sum<V / 2, OFF / 2>(q, lane);
#pragma unroll
        for (int i = 0; i < V / 2; ++i) p[i] = q[i];
    } else {
#pragma unroll
        for (int off = OFF; off >= 1; off >>= 1) p[0] += __shfl_xor(p[0], off, 64);
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

// k_gemv_fused: k_gemv_reg with the rotate + quantize prologue inside.  The row's own loads go out first and the
// first group's weight loads right behind them; while the weights are in flight the workgroup rotates and quantizes
// the activation row (the same per-chunk code as the stand-alone quantizer, so the codes and scales are
// bit-identical), parks the codes in LDS and every lane picks up its share.  One launch per linear instead of two.
// ROT = false: the row arrives in the rotated basis and is only quantized.
// NORM: the row is first normalized, v = ((x (+ res)) * r) * g with r = 1 / sqrt(mean((x + res)^2) + eps), the
// arithmetic of the stand-alone RMSNorm + quantize kernel; workgroup 0 also leaves the residual sum (h_out) and, on
// request, the normalized row (xn_out) for the caller.
struct FusedNorm {
    const float *res, *g;
    float *h_out, *xn_out;
    float eps;
};

template <int CW, int CQ, bool NORM, bool ROT>
__global__ __launch_bounds__(256) void k_gemv_fused(const float *__restrict__ x, const int8_t *__restrict__ qw,
                                                    const float *__restrict__ sw, float *__restrict__ y,
                                                    int8_t *__restrict__ qx_out, float *__restrict__ sx_out, int N,
                                                    int K, FusedNorm nm)
{
    constexpr int BLOCK = 128, LPB = BLOCK / 8;
    constexpr int R = (16 / CW) < 1 ? 1 : (16 / CW);   // rows per wave
    constexpr int V = pow2_ceil(R);
    extern __shared__ __attribute__((aligned(16))) char s_dyn[];
    int8_t *s_x = reinterpret_cast<int8_t *>(s_dyn);            // [K] codes
    float *s_max = reinterpret_cast<float *>(s_dyn + K);        // [4] row maxima, then [4 * CQ] sums of squares
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    constexpr int rows_per_wg = 4 * R;
    // the workgroup owns a run of consecutive groups of rows_per_wg weight rows (the groups dealt out evenly over
    // the grid): one prologue serves them all
    const int ngroups = (N + rows_per_wg - 1) / rows_per_wg;
    const int g0 = (int)((int64_t)ngroups * blockIdx.x / gridDim.x);
    const int g1 = (int)((int64_t)ngroups * (blockIdx.x + 1) / gridDim.x);
    const int kbase = lane * 16;

    auto load_w = [&](v4i (&w)[R][CW], int g) {
        const int row0 = g * rows_per_wg + wave * R;
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int c = 0; c < CW; ++c) {
                const int off = kbase + c * 1024;
                w[r][c] = (row0 + r < N && off < K) ? *reinterpret_cast<const v4i *>(qw + (int64_t)(row0 + r) * K + off)
                                                    : (v4i){0, 0, 0, 0};
            }
    };
    // Loads return in the order they were issued: the first row's own loads (activations, residual, gain) go out
    // BEFORE the first group's weights, so that the prologue's arithmetic runs while the weights are on their way
    // (issued behind them, the row would arrive only after 64 KB of weights per workgroup, and nothing would be in
    // flight while the prologue computes).
    v4i w[R][CW];

    // rotate + quantize: thread t owns chunks t, t + 256, ... of the row
    const int j = tid % LPB;
    const int nchunk = K / 8;
    float v[CQ][8];
    int base[CQ];
#pragma unroll
    for (int i = 0; i < CQ; ++i) {
        const int c = tid + i * 256;
        base[i] = (c / LPB) * BLOCK + 4 * j;
        if (c < nchunk) {
            const float4 lo = *reinterpret_cast<const float4 *>(x + base[i]);
            const float4 hi = *reinterpret_cast<const float4 *>(x + base[i] + BLOCK / 2);
            v[i][0] = lo.x; v[i][1] = lo.y; v[i][2] = lo.z; v[i][3] = lo.w;
            v[i][4] = hi.x; v[i][5] = hi.y; v[i][6] = hi.z; v[i][7] = hi.w;
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[i][e] = 0.0f;
        }
    }
    const bool keeper = blockIdx.x == 0;   // one workgroup also leaves the codes and scales in the caller's workspace
    if constexpr (!NORM) load_w(w, g0);
    if constexpr (NORM) {
        float4 gl[CQ], gh[CQ], rl_[CQ], rh_[CQ];
        float ss[CQ];   // per chunk, then per group of 64 chunks (group wave + 4 * i): the order of fwht_core.h
#pragma unroll
        for (int i = 0; i < CQ; ++i) {
            if (tid + i * 256 < nchunk) {
                gl[i] = *reinterpret_cast<const float4 *>(nm.g + base[i]);
                gh[i] = *reinterpret_cast<const float4 *>(nm.g + base[i] + BLOCK / 2);
                if (nm.res) {
                    const float *rr = nm.res + base[i];
                    rl_[i] = *reinterpret_cast<const float4 *>(rr);
                    rh_[i] = *reinterpret_cast<const float4 *>(rr + BLOCK / 2);
                }
            }
        }
        load_w(w, g0);
#pragma unroll
        for (int i = 0; i < CQ; ++i) {
            ss[i] = 0.0f;
            if (tid + i * 256 < nchunk) {
                if (nm.res) {
                    const float4 rl = rl_[i], rh = rh_[i];
                    v[i][0] = v[i][0] + rl.x; v[i][1] = v[i][1] + rl.y; v[i][2] = v[i][2] + rl.z; v[i][3] = v[i][3] + rl.w;
                    v[i][4] = v[i][4] + rh.x; v[i][5] = v[i][5] + rh.y; v[i][6] = v[i][6] + rh.z; v[i][7] = v[i][7] + rh.w;
                    if (keeper) {
                        float *ho = nm.h_out + base[i];
                        *reinterpret_cast<float4 *>(ho) = make_float4(v[i][0], v[i][1], v[i][2], v[i][3]);
                        *reinterpret_cast<float4 *>(ho + BLOCK / 2) = make_float4(v[i][4], v[i][5], v[i][6], v[i][7]);
                    }
                }
                ss[i] = chunk_sumsq(v[i]);
            }
        }
#pragma unroll
        for (int i = 0; i < CQ; ++i) ss[i] = group_sum(ss[i]);
        if (lane == 0) {
#pragma unroll
            for (int i = 0; i < CQ; ++i) s_max[4 + wave + 4 * i] = ss[i];
        }
        __syncthreads();
        const float total = tree_sum<4 * CQ>(s_max + 4);
        const float r = 1.0f / sqrtf(total / (float)K + nm.eps);
#pragma unroll
        for (int i = 0; i < CQ; ++i) {
            if (tid + i * 256 < nchunk) {
                v[i][0] = (v[i][0] * r) * gl[i].x; v[i][1] = (v[i][1] * r) * gl[i].y;
                v[i][2] = (v[i][2] * r) * gl[i].z; v[i][3] = (v[i][3] * r) * gl[i].w;
                v[i][4] = (v[i][4] * r) * gh[i].x; v[i][5] = (v[i][5] * r) * gh[i].y;
                v[i][6] = (v[i][6] * r) * gh[i].z; v[i][7] = (v[i][7] * r) * gh[i].w;
                if (keeper && nm.xn_out) {
                    float *xo = nm.xn_out + base[i];
                    *reinterpret_cast<float4 *>(xo) = make_float4(v[i][0], v[i][1], v[i][2], v[i][3]);
                    *reinterpret_cast<float4 *>(xo + BLOCK / 2) = make_float4(v[i][4], v[i][5], v[i][6], v[i][7]);
                }
            }
        }
    }
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < CQ; ++i) {
        if constexpr (ROT) fwht_chunk<BLOCK>(v[i], j);   // !ROT: the row arrives in the rotated basis
        amax = fmaxf(amax, abs8(v[i]));
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));
    if (lane == 0) s_max[wave] = amax;
    __syncthreads();
    const float a = fmaxf(fmaxf(s_max[0], s_max[1]), fmaxf(s_max[2], s_max[3]));
    const float sc = (a == 0.0f) ? 1.0f : a / 127.0f;
    const float inv = (a == 0.0f) ? 0.0f : 127.0f / a;
    if (keeper && tid == 0) *sx_out = sc;
#pragma unroll
    for (int i = 0; i < CQ; ++i) {
        if (tid + i * 256 < nchunk) {
            const uint32_t c0 = quant4(v[i][0], v[i][1], v[i][2], v[i][3], inv);
            const uint32_t c1 = quant4(v[i][4], v[i][5], v[i][6], v[i][7], inv);
            *reinterpret_cast<uint32_t *>(s_x + base[i]) = c0;
            *reinterpret_cast<uint32_t *>(s_x + base[i] + BLOCK / 2) = c1;
            if (keeper) {
                *reinterpret_cast<uint32_t *>(qx_out + base[i]) = c0;
                *reinterpret_cast<uint32_t *>(qx_out + base[i] + BLOCK / 2) = c1;
            }
        }
    }
    __syncthreads();

    v4i xr[CW];
#pragma unroll
    for (int c = 0; c < CW; ++c) {
        const int off = kbase + c * 1024;
        xr[c] = off < K ? *reinterpret_cast<const v4i *>(s_x + off) : (v4i){0, 0, 0, 0};
    }
    constexpr int SH = 6 - __builtin_ctz(V);
    const int vi = lane >> SH;
    const bool speaker = (lane & ((1 << SH) - 1)) == 0;
#pragma unroll 1
    for (int g = g0; g < g1; ++g) {
        // the next group's weight loads go out before this group's arithmetic
        v4i wn[R][CW];
        const bool more = g + 1 < g1;   // the same for every thread of the workgroup
        if (more) load_w(wn, g + 1);
        int p[V];
#pragma unroll
        for (int i = 0; i < V; ++i) p[i] = 0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            int a = 0;
#pragma unroll
            for (int c = 0; c < CW; ++c) {
                a = __builtin_amdgcn_sdot4(w[r][c][0], xr[c][0], a, false);
                a = __builtin_amdgcn_sdot4(w[r][c][1], xr[c][1], a, false);
                a = __builtin_amdgcn_sdot4(w[r][c][2], xr[c][2], a, false);
                a = __builtin_amdgcn_sdot4(w[r][c][3], xr[c][3], a, false);
            }
            p[r] = a;
        }
        fold_sum<V, 32>(p, lane);
        const int n = g * rows_per_wg + wave * R + vi;
        if (speaker && vi < R && n < N) y[n] = ((float)p[0] * sc) * sw[n];
        if (more) {
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int c = 0; c < CW; ++c) w[r][c] = wn[r][c];
        }
    }
}

template <int CW, int CQ, bool NORM, bool ROT = true>
static int32_t launch_fused(const float *x, const int8_t *qw, const float *sw, float *y, int8_t *qx, float *sx, int N, int K,
                            const FusedNorm &nm, hipStream_t s)
{
    constexpr int R = (16 / CW) < 1 ? 1 : (16 / CW);
    const size_t lds = (size_t)K + (4 + 4 * CQ) * sizeof(float);   // at most 4,144 bytes
    // Every workgroup reads the whole activation row (with the norm: the residual and the gain too, 48 KB at
    // K = 4096) before its first dot product.  Beyond two workgroups per compute unit a workgroup therefore takes
    // several groups of rows in turn, the next group's weights on their way while it works on the current one.
    constexpr int rows_per_wg = 4 * R;
    const int ngroups = (N + rows_per_wg - 1) / rows_per_wg;
    const unsigned grid = (unsigned)std::min(ngroups, 2 * compute_units());   // three per unit measured the same
    hipLaunchKernelGGL((k_gemv_fused<CW, CQ, NORM, ROT>), dim3(grid), dim3(256), lds, s, x, qw, sw, y, qx, sx, N, K, nm);
    return launch_status();
}

// The fused decode linear is taken for one token and K <= 4096 only (MI_EINVAL tells the caller to take the
// two-kernel path).  Measured: 9.3 against 10.6 us for 4096 -> 6144 at M = 1, but every workgroup repeats the
// quantization, which at M = 4 or K = 14336 costs more than the launch it saves (15.6 against 11.7 us, 20.8
// against 18.8 us).  rotate = false: x is already in the rotated basis (the attention output as the merge leaves
// it) and is only quantized.
int32_t launch_linear_fused(const float *x, const int8_t *qw, const float *sw, float *y, int8_t *qx, float *sx,
                            int64_t M64, int64_t N64, int64_t K64, hipStream_t s, bool rotate)
{
    const int N = (int)N64, K = (int)K64;
    if (M64 != 1 || K % 1024) return MI_EINVAL;
    const int nchunk = K >> 10;
    const FusedNorm none = {nullptr, nullptr, nullptr, nullptr, 0.0f};
    if (rotate) {
        if (nchunk == 4) return launch_fused<4, 2, false>(x, qw, sw, y, qx, sx, N, K, none, s);   // K = 4096
        if (nchunk == 2) return launch_fused<2, 1, false>(x, qw, sw, y, qx, sx, N, K, none, s);   // K = 2048
    } else {
        if (nchunk == 4) return launch_fused<4, 2, false, false>(x, qw, sw, y, qx, sx, N, K, none, s);
        if (nchunk == 2) return launch_fused<2, 1, false, false>(x, qw, sw, y, qx, sx, N, K, none, s);
    }
    return MI_EINVAL;
}

// The same with the (residual +) RMSNorm ahead of the quantizer: one launch for norm + quantize + GEMV of one token.
int32_t launch_norm_linear_fused(const float *x, const float *res, const float *g, float eps, float *h_out,
                                 float *xn_out, const int8_t *qw, const float *sw, float *y, int8_t *qx, float *sx,
                                 int64_t M64, int64_t N64, int64_t K64, hipStream_t s)
{
    const int N = (int)N64, K = (int)K64;
    if (M64 != 1 || K % 1024) return MI_EINVAL;
    const int nchunk = K >> 10;
    const FusedNorm nm = {res, g, h_out, xn_out, eps};
    if (nchunk == 4) return launch_fused<4, 2, true>(x, qw, sw, y, qx, sx, N, K, nm, s);
    if (nchunk == 2) return launch_fused<2, 1, true>(x, qw, sw, y, qx, sx, N, K, nm, s);
    return MI_EINVAL;
}

template <int MB, int CW, int WG, bool DEQ>
static int32_t launch_reg(const int8_t *qx, const float *sx, const int8_t *qw, const float *sw, int32_t *acc,
                          float *y, int M, int N, int K, int QW, hipStream_t s)
{
    constexpr int R = (16 / CW) < 1 ? 1 : (16 / CW);
    const int rows_per_wg = (WG / QW) * R;
    const unsigned grid = (unsigned)((N + rows_per_wg - 1) / rows_per_wg);
    hipLaunchKernelGGL((k_gemv_reg<MB, CW, WG, DEQ>), dim3(grid), dim3(64 * WG), 0, s, qx, qw, sx, sw, acc, y, M, N, K, QW);
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
