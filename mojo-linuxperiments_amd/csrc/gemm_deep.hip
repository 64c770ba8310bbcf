// W8A8 contraction for everything between the GEMV's few tokens and the sizes that fill the chip with 256-wide tiles:
//   acc[m,n] = sum_k qx[m,k] * qw[n,k],   y = ((float)acc * sx[m]) * sw[n]
//
// One workgroup per tile, the tile chosen from sixteen (16 x 16 to 192 x 128) so that every compute
// unit has one, and one load stream per workgroup: stages of 128 to 512 bytes of K go straight to LDS through a ring of D
// buffers, D - 1 stages in flight, one barrier a stage.  The tiles of 128 columns, 128 x 96, 128 x 64 and 32 x 48 take more than half
// of a unit's LDS, the others at most half: where there are tiles enough two workgroups share a unit and hide each other's first loads and last stores (16 rows,
// 4096 -> 28672 inside a decode step: 24.3 instead of 27.2 us).  Small tiles leave most
// waves without rows of their own, so the waves split K inside a stage (WK slices of 64 bytes) and meet once, through
// LDS, at the tile's end; every wave finishes an equal share of the matrix-instruction tiles.
//
// Four or eight waves multiply and four more only load: they request a stage, wait until an older one has landed and say so
// by the barrier.  A load holds its wave's issue until the path to the cache takes it, and with the loads dealt to the
// multiplying waves the matrix instructions behind them waited for that path: a stage of a 128 x 128 tile alone on the
// chip took 0.33 us, 0.29 with loading waves (512 clocks of matrix instructions, 32 loads at 16 clocks).  With the two
// halves of the multiplying waves a phase apart: 0.33 without loading waves, 0.29 with them.  One or two loading waves measured
// the same at large tiles and 0.1 to 0.2 us more at small ones, whose first loads they request one by one; eight mixed.
//
// What bounds it.  Few rows: HBM and launch to first byte.  128 x 128 tiles on a full chip: 0.39 us a stage, which falls to 0.34 with codes
// that are all zero (the part's power limit), is the same with two, three or four stages in flight (not latency), and
// of which the path to the cache takes 0.25 (130 GB/s a unit in a loop of nothing but loads).  So the tile decides: rows loaded per result.
//
// Measured (us a call in a graph of them, weights from HBM, and with the loads made by the waves that multiply):
// 8 x 1408 -> 736 2.78 (3.00), 16 x 4096 -> 6144 7.14 (7.36), 32 x 4096 -> 4096 6.28 (6.51), 64 x 4096 -> 14336 15.2 (15.6),
// 97 x 4096 -> 4096 8.12 (8.67), 168 x 2944 -> 2320 5.38 (6.18), 200 x 4096 -> 14336 23.6 (24.3), 256 x 14336 -> 4096 34.5 (34.5),
// 397 x 3072 -> 7136 17.7 (18.4), 925 x 1664 -> 2784 10.7 (11.6), 1007 x 3456 -> 1296 10.8 (11.6); 16 x 4096 -> 28672 23.9 (23.9).
//
// LDS layout, swizzle and shape of the loads are those of gemm_tiled.hip: 1 KB blocks of 8 rows x 128 bytes, chunk position
// XORed with sigma(row, block parity), free of bank conflicts for the fragment reads.  Operand A is the weights.
//
#include <algorithm>
#include <utility>
#include <vector>

#include "common.h"
#include "gemm_deep.h"
#include "lds_ops.h"

namespace mi {
namespace deep {

typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));   // four scales: a batch asks only 4 bytes of alignment of them


template <int TM_, int TN_, int WM_, int WN_, int WK_, int D_>
struct Cfg {
    static constexpr int TM = TM_, TN = TN_, WM = WM_, WN = WN_, WK = WK_, D = D_;
    static constexpr int NW = WM * WN * WK, NL = 4, TPB = 64 * (NW + NL);   // waves that multiply, waves that load
    static constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN;
    static constexpr int SUB = WK / 2;                  // 128-byte K steps per stage
    static constexpr int BX = BM / 8, BW = BN / 8;      // 1 KB blocks (8 rows x 128 B) per step
    static constexpr int BLK = (BX + BW) * SUB;         // per stage
    static constexpr int L = BLK / NL;                  // load instructions per loading wave and stage
    static constexpr int STAGE = BLK * 1024;
    static constexpr int NF = TM * TN;                  // matrix-instruction tiles of a wave
    static constexpr int OWN = (NF + WK - 1) / WK;      // of which it finishes this many (the last waves fewer or none)
    static constexpr int PART = WM * WN * NF * (WK - 1) * 1024;
    static constexpr int LDS = D * STAGE > PART ? D * STAGE : PART;
    static constexpr bool PAIR = OWN % 2 == 0 && TN % 2 == 0 && NF % OWN == 0;
    static_assert(WK % 2 == 0 && BLK % NL == 0 && LDS <= 160 * 1024, "");
    static_assert((D - 1) * L < 60 && D >= 2 && D <= 7, "vmcnt counts to 63");
};

// A loading wave (`w` of NL): all stages of the tile, in step with the multiplying waves' barriers
template <typename C>
__device__ __forceinline__ void load_stages(const int8_t *__restrict__ qx, const int8_t *__restrict__ qw, const int M, const int N,
                                            const int K, const int m0, const int n0, char *smem, const int w, const int lane)
{
    constexpr int D = C::D, SUB = C::SUB, L = C::L;
    const int nk = K >> 7, ns = (nk + SUB - 1) / SUB;
    // load i fills block b = w + NL * i of a stage; lane l = 8 * rho + c fetches chunk c ^ sigma of row rho
    const int8_t *base[L];
    unsigned roff[L];
    int sub[L];
    {
        const int rho = lane >> 3, c = lane & 7;
        const int8_t *const xt = qx + (int64_t)m0 * K, *const wt = qw + (int64_t)n0 * K;
#pragma unroll
        for (int i = 0; i < L; ++i) {
            const int b = w + C::NL * i;
            sub[i] = SUB == 1 ? 0 : b / (C::BX + C::BW);
            const int rb = b - sub[i] * (C::BX + C::BW);
            const bool isx = rb < C::BX;
            const int blk = isx ? rb : rb - C::BX;
            const int sigma = ((blk & 1) << 2) | (rho >> 1);
            const int row = min(blk * 8 + rho, isx ? M - 1 - m0 : N - 1 - n0);   // rows past the edge repeat the last one
            base[i] = isx ? xt : wt;
            roff[i] = (unsigned)row * (unsigned)K + (unsigned)((c ^ sigma) << 4);
        }
    }
    const unsigned lds0 = (unsigned)(uintptr_t)(lptr_t)smem + w * 1024;
    auto issue = [&](int s, unsigned buf) {
#pragma unroll
        for (int i = 0; i < L; ++i) {
            int k = s * SUB + sub[i];
            if (SUB > 1 && k > nk - 1) k = nk - 1;   // a last stage that is not whole: its steps past K are not used
            dma16(base[i], roff[i] + (unsigned)(k << 7), lds0 + buf + i * C::NL * 1024);
        }
    };
    // at most the loads of the `behind` stages issued after it may be in flight: a stage has landed (this wave's share)
    auto landed = [&](int behind) {   // wave-uniform, below D - 1
        if (D > 2 && behind == D - 2) wait_vm<(D > 2 ? D - 2 : 0) * L>();
        else if (D > 3 && behind == D - 3) wait_vm<(D > 3 ? D - 3 : 0) * L>();
        else if (D > 4 && behind == D - 4) wait_vm<(D > 4 ? D - 4 : 0) * L>();
        else if (D > 5 && behind == D - 5) wait_vm<(D > 5 ? D - 5 : 0) * L>();
        else wait_vm<0>();
    };
#pragma unroll
    for (int s = 0; s < D - 1; ++s)
        if (s < ns) issue(s, s * C::STAGE);
    landed(min(ns, D - 1) - 1);
    __builtin_amdgcn_s_barrier();   // the first stage has landed
    unsigned buf = (D - 1) * C::STAGE;
    int s = 0;
    for (; s + D - 1 < ns; ++s) {   // the multiplying waves read stage s
        issue(s + D - 1, buf);      // into the buffer of stage s - 1
        buf = buf + C::STAGE == D * C::STAGE ? 0 : buf + C::STAGE;
        wait_vm<(D - 2) * L>();
        __builtin_amdgcn_s_barrier();   // stage s + 1 has landed and everybody holds stage s in registers
    }
    for (; s < ns; ++s) {
        if (s + 1 < ns) landed(ns - 2 - s);
        __builtin_amdgcn_s_barrier();
    }
}

template <typename C, bool DEQ>
__device__ __forceinline__ void tile(const int8_t *__restrict__ qx, const int8_t *__restrict__ qw, const float *__restrict__ sx,
                                     const float *__restrict__ sw, void *__restrict__ out, const int M, const int N, const int K,
                                     const int m0, const int n0, char *smem)
{
    constexpr int TM = C::TM, TN = C::TN, WK = C::WK, D = C::D, SUB = C::SUB, OWN = C::OWN;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nk = K >> 7, ns = (nk + SUB - 1) / SUB;

    if (wave >= C::NW) {
        load_stages<C>(qx, qw, M, N, K, m0, n0, smem, wave - C::NW, lane);
        __syncthreads();   // the two at the tile's end
        __syncthreads();
        return;
    }

    // read side: wave (wm, wn, wk) multiplies K half wk % 2 of step wk / 2 of every stage
    const int wk = wave % WK, wmn = wave / WK;
    const int wm = wmn % C::WM, wn = wmn / C::WM;
    const int r = lane & 15, g = lane >> 4;
    const char *xa, *wa;
    {
        const int rho = r & 7, par = r >> 3, sigma = (par << 2) | (rho >> 1);
        const int off = par * 1024 + ((8 * rho + ((4 * (wk & 1) + g) ^ sigma)) << 4);
        const char *st = smem + (wk >> 1) * (C::BX + C::BW) * 1024 + off;
        xa = st + wm * TM * 2048;
        wa = st + C::BX * 1024 + wn * TN * 2048;
    }
    struct Frags {
        v4i x[TM], w[TN];
    };
    auto fetch = [&](Frags &f, unsigned buf) {
#pragma unroll
        for (int i = 0; i < TM; ++i) f.x[i] = *reinterpret_cast<const v4i *>(xa + buf + i * 2048);
#pragma unroll
        for (int j = 0; j < TN; ++j) f.w[j] = *reinterpret_cast<const v4i *>(wa + buf + j * 2048);
    };

    // tile f = i * TN + j of a wave is finished by the wave of K slice f / OWN; its scales are requested here
    const int f0 = wk * OWN;
    const int mw = m0 + wm * TM * 16, nw = n0 + wn * TN * 16;
    const bool lo = r < 8;
    float sxv[OWN];
    f4u swv[OWN];
    if constexpr (DEQ) {
#pragma unroll
        for (int o = 0; o < OWN; ++o) {
            const int f = min(f0 + o, C::NF - 1), i = f / TN, j = f % TN;
            if constexpr (C::PAIR) {   // of an even and an odd tile side by side, see the stores
                const int m = mw + i * 16 + (o & 1) * 8 + (r & 7), n = nw + (j & ~1) * 16 + (lo ? 0 : 16) + 4 * g;
                sxv[o] = sx[min(m, M - 1)];
                if (!(o & 1)) swv[o] = *reinterpret_cast<const f4u *>(sw + min(n, N - 4));
            } else {
                const int m = mw + i * 16 + r, n = nw + j * 16 + 4 * g;
                sxv[o] = sx[min(m, M - 1)];
                swv[o] = *reinterpret_cast<const f4u *>(sw + min(n, N - 4));
            }
        }
    }

    v4i acc[C::NF];
#pragma unroll
    for (int f = 0; f < C::NF; ++f) acc[f] = (v4i){0, 0, 0, 0};

    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    Frags f;
    unsigned cur = 0;
    for (int s = 0; s < ns; ++s) {
        fetch(f, cur);
        __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0), as an instruction that the compiler's own counting sees
        if (SUB == 1 || s * SUB + (wk >> 1) < nk) {
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int i = 0; i < TM; ++i)
                    acc[i * TN + j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(f.w[j], f.x[i], acc[i * TN + j], 0, 0, 0);
        }
        __builtin_amdgcn_s_barrier();   // as in load_stages
        asm volatile("" ::: "memory");
        cur = cur + C::STAGE == D * C::STAGE ? 0 : cur + C::STAGE;
    }
    __syncthreads();

    // the K slices meet: every wave hands the tiles it does not finish to the wave that does, [wmn][tile][slice][lane]
    char *const part = smem + wmn * C::NF * (WK - 1) * 1024 + lane * 16;
#pragma unroll
    for (int f = 0; f < C::NF; ++f) {
        const int own = f / OWN;
        if (own != wk) *reinterpret_cast<v4i *>(part + (f * (WK - 1) + (wk < own ? wk : wk - 1)) * 1024) = acc[f];
    }
    __syncthreads();
    if (f0 >= C::NF) return;
    v4i sum[OWN];
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
#pragma unroll
        for (int w = 0; w < WK; ++w)
            if (w == wk) sum[o] = acc[w * OWN + o < C::NF ? w * OWN + o : 0];
        const int f = min(f0 + o, C::NF - 1);
#pragma unroll
        for (int w = 0; w < WK - 1; ++w) sum[o] += *reinterpret_cast<const v4i *>(part + (f * (WK - 1) + w) * 1024);
    }
    // a lane holds channels 4 g .. + 3 of token r of a tile
    auto put = [&](const v4i &v, float sxm, const f4u &s4, int m, int n) {
        if (m >= M || n >= N) return;
        const int64_t at = (int64_t)m * N + n;
        if constexpr (DEQ) {
            float4 o;
            o.x = ((float)v[0] * sxm) * s4.x;
            o.y = ((float)v[1] * sxm) * s4.y;
            o.z = ((float)v[2] * sxm) * s4.z;
            o.w = ((float)v[3] * sxm) * s4.w;
            *reinterpret_cast<float4 *>(static_cast<float *>(out) + at) = o;
        } else {
            *reinterpret_cast<v4i *>(static_cast<int32_t *>(out) + at) = v;
        }
    };
    if constexpr (C::PAIR) {
        // two tiles side by side trade halves between lanes r and r ^ 8: one store writes 8 rows x 128 bytes
#pragma unroll
        for (int o = 0; o < OWN; o += 2) {
            const int i = (f0 + o) / TN, j = (f0 + o) % TN;
            v4i t0, t1;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                t0[e] = ror8(sum[o][e]);
                t1[e] = ror8(sum[o + 1][e]);
            }
            const int m = mw + i * 16 + (r & 7), n = nw + j * 16 + (lo ? 0 : 16) + 4 * g;
            put(lo ? sum[o] : t1, sxv[o], swv[o], m, n);
            put(lo ? t0 : sum[o + 1], sxv[o + 1], swv[o], m + 8, n);
        }
    } else {
#pragma unroll
        for (int o = 0; o < OWN; ++o) {
            if (f0 + o >= C::NF) break;
            const int i = (f0 + o) / TN, j = (f0 + o) % TN;
            put(sum[o], sxv[o], swv[o], mw + i * 16 + r, nw + j * 16 + 4 * g);
        }
    }
}

// A grid's threads in one direction stay below 2^32: more workgroups than 2^ROW_LOG2 lie in rows of that many, the last one not whole.
constexpr int ROW_LOG2 = 22;

// Tile of workgroup `id` of a problem (ids go round robin over the XCDs): an XCD takes an eighth of the tiles, column by
// column, so that the row tiles of a weight column meet in its L2 and no XCD has a tile more than another.
// magic = ceil(2^32 / tiles_m) divides exactly: tiles * tiles_m < 2^32.
__device__ __forceinline__ bool tile_of(int id, int tiles, int tiles_m, unsigned magic, int *tm, int *tn)
{
    const unsigned x = (unsigned)id & 7, t = (((unsigned)tiles * x) >> 3) + ((unsigned)id >> 3);
    *tn = tiles_m == 1 ? (int)t : (int)__umulhi(t, magic);
    *tm = (int)t - *tn * tiles_m;
    return t < ((unsigned)tiles * (x + 1)) >> 3;
}

template <typename C, bool DEQ>
__global__ __launch_bounds__(C::TPB) void k_w8a8_deep(const int8_t *__restrict__ qx, const int8_t *__restrict__ qw, int M, int N,
                                                      int K, int tiles, int tiles_m, unsigned magic,
                                                      const float *__restrict__ sx, const float *__restrict__ sw,
                                                      void *__restrict__ out)
{
    extern __shared__ __attribute__((aligned(16))) char smem[];
    int tm, tn;
    if (!tile_of((int)(blockIdx.x + (blockIdx.y << ROW_LOG2)), tiles, tiles_m, magic, &tm, &tn)) return;
    tile<C, DEQ>(qx, qw, sx, sw, out, M, N, K, tm * C::BM, tn * C::BN, smem);
}

// false: more tiles than the kernel's arithmetic covers
static bool tile_grid(int bm, int bn, int M, int N, int *tiles, int *tiles_m, unsigned *magic)
{
    const int64_t tm = ((int64_t)M + bm - 1) / bm, all = tm * (((int64_t)N + bn - 1) / bn);
    if (all > (1 << 24) || all * tm >= (1ll << 32)) return false;
    *tiles = (int)all;
    *tiles_m = (int)tm;
    *magic = (unsigned)(((1ull << 32) + (unsigned long long)tm - 1) / (unsigned long long)tm);
    return true;
}

// several contractions in one launch, workgroups of the first problem first
struct Batch {
    DeepProblem p[DEEP_MAX];
    int n;
};
template <typename C, bool DEQ>
__global__ __launch_bounds__(C::TPB) void k_w8a8_deep_batch(const Batch b)
{
    extern __shared__ __attribute__((aligned(16))) char smem[];
    int pi = 0;
#pragma unroll
    for (int k = 1; k < DEEP_MAX; ++k)
        if (k < b.n && (int)blockIdx.x >= b.p[k].first) pi = k;
    const DeepProblem &P = b.p[pi];
    int tm, tn;   // (P.first % 8 == 0)
    if (!tile_of((int)blockIdx.x - P.first, P.tiles, P.tiles_m, P.magic, &tm, &tn)) return;
    tile<C, DEQ>(P.qx, P.qw, P.sx, P.sw, P.out, P.M, P.N, P.K, tm * C::BM, tn * C::BN, smem);
}

template <typename C, bool DEQ>
static int32_t launch_batch(Batch &b, hipStream_t s)
{
    int64_t grid = 0;
    for (int i = 0; i < b.n; ++i) {
        DeepProblem &p = b.p[i];
        if (p.M <= 0 || p.N <= 0 || p.N % 16 || p.K < 128 || p.K % 128) return MI_EINVAL;
        if (!tile_grid(C::BM, C::BN, p.M, p.N, &p.tiles, &p.tiles_m, &p.magic)) return MI_ERANGE;
        p.first = (int)grid;
        grid += (p.tiles + 7) / 8 * 8;
        if (grid > 0x7fffffff / C::TPB) return MI_ERANGE;
    }
    MI_LDS_OPT_IN((&k_w8a8_deep_batch<C, DEQ>), C::LDS);
    launch_kernel((k_w8a8_deep_batch<C, DEQ>), dim3((unsigned)grid), dim3(C::TPB), C::LDS, s, b);
    return launch_status();
}

template <typename C, bool DEQ>
static int32_t launch(const int8_t *qx, const float *sx, const int8_t *qw, const float *sw, void *out, int M, int N, int K,
                      hipStream_t s)
{
    // ragged M and N are the kernel's to clamp; it moves whole 128-byte K steps and stores whole 16-column groups
    if (M <= 0 || N <= 0 || N % 16 || K < 128 || K % 128) return MI_EINVAL;
    MI_LDS_OPT_IN((&k_w8a8_deep<C, DEQ>), C::LDS);
    int tiles, tiles_m;
    unsigned magic;
    if (!tile_grid(C::BM, C::BN, M, N, &tiles, &tiles_m, &magic)) return MI_ERANGE;
    constexpr unsigned ROW = 1u << ROW_LOG2;
    static_assert((uint64_t)ROW * C::TPB < (1ull << 32) && ROW % 8 == 0, "");
    const unsigned wgs = (unsigned)(tiles + 7) / 8 * 8;
    launch_kernel((k_w8a8_deep<C, DEQ>), wgs <= ROW ? dim3(wgs) : dim3(ROW, (wgs + ROW - 1) / ROW), dim3(C::TPB), C::LDS, s, qx, qw,
                  M, N, K, tiles, tiles_m, magic, sx, sw, out);
    return launch_status();
}

// ---- which tile ----------------------------------------------------------------------------------------------------
// Time of a launch in microseconds, fitted to 250 shapes (M of 2 to 1024, N of 784 to 28672, K of 1024 to 14336) times
// every tile, each measured behind the quantizer that feeds it and with weights from HBM.  A unit moves (BM + BN) * 128
// bytes per K step through its load path at 1.69 ns a row (76 GB/s, 28 clocks a KB: as it was when the waves that multiply made the
// loads; with waves of their own a launch takes 2 to 6 % less, and the figures stay for the order of the tiles that they give), 1.82
// instead of 2 times as long
// for two workgroups side by side, and pays 0.7 us plus the tile's outputs per round of tiles.  The memory's share,
// bytes at 5 TB/s, is joined as a 4-norm: it does not depend on the tile.  Over 1059 drawn shapes of 129 to 1024 rows the choice that rests
// on it takes 1.061 of the time of the best of all tiles and kernels, with the finer estimate below 1.016.
struct Tile {
    int bm, bn, sub, per_cu;
};
constexpr Tile TILES[] = {{128, 128, 1, 1}, {128, 64, 1, 1}, {64, 64, 1, 2},  {64, 32, 1, 2},  {32, 48, 2, 1},
                          {32, 32, 2, 2},   {32, 16, 2, 2},  {16, 48, 2, 2},  {16, 32, 2, 2},  {16, 16, 4, 2},
                          {160, 128, 1, 1}, {96, 128, 1, 1}, {128, 96, 1, 1}, {192, 128, 1, 1}, {96, 64, 1, 2}, {64, 96, 1, 2}};
constexpr int COARSE = 10;   // tiles that pick() knows
constexpr float PER_LAUNCH = 1.72f, PER_ROUND = 0.68f, PER_OUTPUT = 2.34e-4f, PER_ROW_STEP = 0.00169f, BESIDE = 0.82f,
                LAST_ROUND = 1.04f, PER_MB = 0.202f;

static inline float alone(const Tile &t, int64_t nk)   // a tile on a unit of its own, without PER_ROUND
{
    return (float)(t.bm * t.bn) * PER_OUTPUT + (float)((nk + t.sub - 1) / t.sub * t.sub) * (float)(t.bm + t.bn) * PER_ROW_STEP;
}

// core time of a tile, without the memory's share (a template: the divisions by its sides are by constants)
template <int I>
static float core_time(int M, int N, int K, int cus)
{
    constexpr Tile t = TILES[I];
    const uint64_t tiles = (uint64_t)(((unsigned)M + t.bm - 1) / t.bm) * (((unsigned)N + t.bn - 1) / t.bn);
    const unsigned slots = (unsigned)(cus * t.per_cu);
    const uint64_t full = tiles >> 32 ? tiles / slots : (unsigned)tiles / slots;
    const unsigned rem = (unsigned)(tiles - full * slots);
    const float one = alone(t, K >> 7), two = (1.0f + BESIDE) * one;
    float c = (float)full * (PER_ROUND + (t.per_cu == 2 ? two : one));
    if (rem) c += (full ? LAST_ROUND : 1.0f) * (PER_ROUND + (rem > (unsigned)cus ? two : one));
    return c;
}
template <int... I>
static void core_times(std::integer_sequence<int, I...>, float *t, int M, int N, int K, int cus)
{
    ((t[I] = core_time<I>(M, N, K, cus)), ...);
}

// core time of the best tile
static float pick(int M, int N, int K, int cus, int *which)
{
    float t[COARSE];
    core_times(std::make_integer_sequence<int, COARSE>{}, t, M, N, K, cus);
    *which = (int)(std::min_element(t, t + COARSE) - t);
    return t[*which];
}

static float with_memory(float core, double bytes)
{
    const float mem = PER_MB * 1e-6f * (float)bytes, c2 = core * core, m2 = mem * mem;
    return PER_LAUNCH + sqrtf(sqrtf(c2 * c2 + m2 * m2));
}

}  // namespace deep

// Microseconds that launch_deep would take, to be compared with the LDS-tiled kernel's; *which is the tile to pass on.  The fit
// above tells tiles apart but not kernels: it is 6 % low on average and 17 % beyond six rounds.  For the tiles that meet the
// other kernel: a constant, a time per round and per K step of a round, which grows with the share of the chip that has a
// tile, and the output; least squares over 2043 of 2600 drawn shapes (M of 65 to 4096, N of 256 to 28672, K of 128 to 14336,
// weights from HBM; standard deviation 6 to 8 %).  Raised by 4 %: near a tie the LDS-tiled kernel is taken, whose own
// estimate is the better one.
float deep_estimate(int M, int N, int K, int cus, int *which)
{
    using namespace deep;
    constexpr float c0[3] = {3.52f, 2.90f, 3.20f}, per_round[3] = {3.09f, 1.25f, 0.31f}, per_step[3] = {0.317f, 0.262f, 0.185f},
                    with_fill[3] = {0.845f, 0.134f, 0.153f}, per_out_mb[3] = {0.067f, 0.242f, 0.200f};
    const float core = pick(M, N, K, cus, which);
    const int w = *which;
    if (w > 2) return 1.06f * with_memory(core, (double)N * K + (double)M * K + 4.0 * M * N);
    const Tile &t = TILES[w];
    const uint64_t tiles = (uint64_t)(((unsigned)M + t.bm - 1) / t.bm) * (((unsigned)N + t.bn - 1) / t.bn);
    const uint64_t slots = (uint64_t)(cus * t.per_cu), full = tiles / slots, rem = tiles - full * slots;
    const float two = 1.0f + BESIDE;   // rounds of one tile a unit
    const float rounds = (float)full * (t.per_cu == 2 ? two : 1.0f) + (rem > (uint64_t)cus ? two : rem ? 1.0f : 0.0f);
    const float fill = (float)tiles / (float)(slots * (full + (rem != 0)));
    const float step = per_step[w] * (1.0f + with_fill[w] * fill * fill);
    return 1.04f * (c0[w] + rounds * (per_round[w] + step * (float)(K >> 7)) + per_out_mb[w] * 4e-6f * (float)M * (float)N);
}

// A finer estimate for 129 to 1024 rows and K from 1024, where a ragged edge or a half-empty round costs most: six more tiles, and
// a constant, a time per K step of a round, which grows with the share of the slots that have a tile, and the output for each tile
// that is worth having there.  Least squares over the times of every tile of 1447 drawn shapes (N of 512 to 28672, K to 14336,
// weights from HBM, behind the quantizer; standard deviation 7 to 8 %, of 1200 others 8 to 10).  Below 129 rows the tiles above are
// within 1 % of the best of all; beyond 1024 no shape was timed.
namespace deep {
struct Fine {
    int tile;
    float c0, step, with_fill, out_mb;
};
constexpr Fine FINE[] = {{0, 3.32f, 0.445f, 0.141f, 0.318f},  {1, 2.51f, 0.312f, 0.133f, 0.344f},  {2, 2.27f, 0.225f, 0.194f, 0.138f},
                         {3, 2.27f, 0.154f, 0.159f, 0.137f},  {5, 2.25f, 0.103f, 0.148f, 0.268f},  {10, 3.67f, 0.496f, 0.069f, 0.347f},
                         {11, 3.07f, 0.407f, 0.159f, 0.259f}, {12, 2.69f, 0.395f, 0.076f, 0.339f}, {13, 3.65f, 0.569f, 0.037f, 0.330f},
                         {14, 2.42f, 0.291f, 0.162f, 0.149f}, {15, 2.31f, 0.300f, 0.241f, 0.115f}};
// (a template, as core_time: the divisions by a tile's sides are by constants.  The choice of a kernel takes the host 190 ns in this
// range and 50 for few rows, 330 and 110 with loops over the tables; a small linear is bound by its host)
template <int I>
static float fine_time(unsigned M, unsigned N, unsigned nk, unsigned cus, float mem4)
{
    constexpr Fine f = FINE[I];
    constexpr Tile t = TILES[f.tile];
    static_assert(t.sub == 1 || t.sub == 2, "");
    constexpr float two = 1.0f + BESIDE;
    const unsigned tiles = ((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
    const unsigned slots = cus * t.per_cu, full = tiles / slots, rem = tiles - full * slots;
    const float rounds = (float)full * (t.per_cu == 2 ? two : 1.0f) + (rem > cus ? two : rem ? 1.0f : 0.0f);
    const float fill = (float)tiles / (float)(slots * (full + (rem != 0)));
    const float steps = (float)(t.sub == 2 ? (nk + 1) & ~1u : nk);
    const float core = rounds * f.step * steps * (1.0f + f.with_fill * fill * fill) + f.out_mb * 4e-6f * (float)M * (float)N, c2 = core * core;
    return f.c0 + sqrtf(sqrtf(c2 * c2 + mem4));
}
constexpr int FINES = (int)(sizeof(FINE) / sizeof(FINE[0]));
template <int... I>
static void fine_times(std::integer_sequence<int, I...>, float *t, unsigned M, unsigned N, unsigned nk, unsigned cus, float mem4)
{
    ((t[I] = fine_time<I>(M, N, nk, cus, mem4)), ...);
}
}  // namespace deep

// The tile to take in place of `coarse`, the choice of deep_estimate, or of the LDS-tiled kernel (coarse < 0) that would take
// `tiled_us`; -1: stay with that kernel.  Another tile has to promise 8 %, as the estimates are good to that: over 1059 drawn
// shapes, weights from HBM, the contraction then takes 0.96 of the time of the coarse choice with 129 to 256 rows, with 257 to 512 and with
// 513 to 1024 (332 of them go over: 0.87); 15 shapes lose more than 3 %, most of them by two rounds of 160 rows in place of one of the
// LDS-tiled kernel (291 x 3072 -> 21984 41.0 -> 46.9).  290 x 4096 -> 14336 34.6 -> 27.9 us, 350 x 4096 -> 6144
// 21.8 -> 17.4, 600 x 4096 -> 4096 21.1 -> 17.9, 1007 x 3456 -> 1296 10.7 -> 9.7.  A lower tile of the same columns of which there are as
// many does not keep that promise where the weights are long: rows past the edge cost the higher one little (they read one row), and its
// ring is the longer.  Of 70 such shapes with K from 2688 the lower one took 1.02 of the time in the mean and up to 1.16 (270 x 6656 ->
// 8288 28.5 -> 31.6, 273 x 5120 -> 5232 17.1 -> 18.6), 1.00 below K = 2560 (of 128 columns) and 5120 (of 64).
int deep_fine(int M, int N, int K, int cus, int coarse, float tiled_us)
{
    using namespace deep;
    if (M <= 128 || M > 1024 || K < 1024 || N > 32768) return coarse;
    const float mem = PER_MB * 1e-6f * ((float)N * (float)K + (float)M * (float)K + 4.0f * (float)M * (float)N), m2 = mem * mem;
    int best = -1;
    float us = 0.0f, now = -1.0f;
    float t[FINES];
    fine_times(std::make_integer_sequence<int, FINES>{}, t, (unsigned)M, (unsigned)N, (unsigned)K >> 7, (unsigned)cus, m2 * m2);
    for (int i = 0; i < FINES; ++i) {
        if (best < 0 || t[i] < us) best = FINE[i].tile, us = t[i];
        if (FINE[i].tile == coarse) now = t[i];
    }
    if (coarse < 0) return 1.08f * us < tiled_us ? best : -1;
    if (K * TILES[best].bn >= 2560 * 128 && TILES[best].bn == TILES[coarse].bn && TILES[best].bm < TILES[coarse].bm &&
        ((unsigned)M + TILES[best].bm - 1) / TILES[best].bm == ((unsigned)M + TILES[coarse].bm - 1) / TILES[coarse].bm)
        return coarse;
    return us < 0.92f * now ? best : coarse;   // (now < 0: a tile for few rows, of few columns)
}

void deep_tile(int which, int32_t *rows, int32_t *cols)
{
    *rows = deep::TILES[which].bm;
    *cols = deep::TILES[which].bn;
}

bool deep_fits(int which, int M, int N)
{
    int tiles, tiles_m;
    unsigned magic;
    return deep::tile_grid(deep::TILES[which].bm, deep::TILES[which].bn, M, N, &tiles, &tiles_m, &magic);
}

template <bool DEQ>
int32_t launch_deep(int which, const int8_t *qx, const float *sx, const int8_t *qw, const float *sw, int32_t *acc, float *y,
                    int64_t M64, int64_t N64, int64_t K64, hipStream_t s)
{
    using namespace deep;
    const int M = (int)M64, N = (int)N64, K = (int)K64;
    void *out = DEQ ? (void *)y : (void *)acc;
    switch (which) {   // in the order of TILES
    case 0: return launch<Cfg<4, 4, 2, 2, 2, 5>, DEQ>(qx, sx, qw, sw, out, M, N, K, s);
    case 1: return launch<Cfg<4, 2, 2, 2, 2, 6>, DEQ>(qx, sx, qw, sw, out, M, N, K, s);
    case 2: return launch<Cfg<2, 2, 2, 2, 2, 5>, DEQ>(qx, sx, qw, sw, out, M, N, K, s);
    case 3: return launch<Cfg<2, 2, 2, 1, 2, 6>, DEQ>(qx, sx, qw, sw, out, M, N, K, s);
    case 4: return launch<Cfg<2, 3, 1, 1, 4, 6>, DEQ>(qx, sx, qw, sw, out, M, N, K, s);
    case 5: return launch<Cfg<2, 2, 1, 1, 4, 5>, DEQ>(qx, sx, qw, sw, out, M, N, K, s);
    case 6: return launch<Cfg<2, 1, 1, 1, 4, 6>, DEQ>(qx, sx, qw, sw, out, M, N, K, s);
    case 7: return launch<Cfg<1, 3, 1, 1, 4, 5>, DEQ>(qx, sx, qw, sw, out, M, N, K, s);
    case 8: return launch<Cfg<1, 2, 1, 1, 4, 6>, DEQ>(qx, sx, qw, sw, out, M, N, K, s);
    case 9: return launch<Cfg<1, 1, 1, 1, 8, 4>, DEQ>(qx, sx, qw, sw, out, M, N, K, s);
    case 10: return launch<Cfg<5, 4, 2, 2, 2, 4>, DEQ>(qx, sx, qw, sw, out, M, N, K, s);
    case 11: return launch<Cfg<3, 4, 2, 2, 2, 5>, DEQ>(qx, sx, qw, sw, out, M, N, K, s);
    case 12: return launch<Cfg<4, 3, 2, 2, 2, 5>, DEQ>(qx, sx, qw, sw, out, M, N, K, s);
    case 13: return launch<Cfg<6, 4, 2, 2, 2, 4>, DEQ>(qx, sx, qw, sw, out, M, N, K, s);
    case 14: return launch<Cfg<3, 2, 2, 2, 2, 4>, DEQ>(qx, sx, qw, sw, out, M, N, K, s);
    case 15: return launch<Cfg<2, 3, 2, 2, 2, 4>, DEQ>(qx, sx, qw, sw, out, M, N, K, s);
    default: return MI_EINVAL;
    }
}
template int32_t launch_deep<true>(int, const int8_t *, const float *, const int8_t *, const float *, int32_t *, float *,
                                   int64_t, int64_t, int64_t, hipStream_t);
template int32_t launch_deep<false>(int, const int8_t *, const float *, const int8_t *, const float *, int32_t *, float *,
                                    int64_t, int64_t, int64_t, hipStream_t);

// ---- several contractions of at least 256 rows in one launch (a part of a batch, see gemm_list.hip)
// Times as above; the tiles go to the units as these come free, longest K first.  A launch of several rounds takes 1.25
// times the sum of its tiles (measured 147 us where the sum says 115 and 83 where it says 66; what the choice that rests on
// it gives over drawn batches stands in gemm_list.hip), one with at most a tile of 160 or 192 rows a unit 1.15 (1.11 and 1.13 in the mean
// of 53; without it 259 x 10240 -> 560 and 4096 -> 13456 took 57 us in such tiles for 41, 259 x 8192 -> 5520 beside 613 x 1152 ->
// 3648 42 for 34).
float deep_batch_estimate(const int64_t *mnk, const int *idx, int n, int cus, int *which)
{
    using namespace deep;
    // 128 x 128, 128 x 64, 64 x 64 and, where the longest K is from 8192 and the shortest from 1024, 160 x 128 and 192 x 128: the four
    // projections with 300 rows 117 -> 101 us, with 384 134 -> 113, with 560 189 -> 167 (quantizer included).  The limits stand in for
    // an estimate that tells batches of shorter K apart, which this one does not: with these tiles there as well 170 drawn batches took
    // 0.93 of the time in the mean, 36 of them more than 1.03 and up to 1.24 of it.
    constexpr int TRY[] = {0, 1, 2, 10, 13};
    const bool finer = mnk[3 * idx[0] + 2] >= 8192 && mnk[3 * idx[n - 1] + 2] >= 1024;
    float best = -1.0f;
    double bytes = 0.0;
    for (int i = 0; i < n; ++i) {
        const double M = (double)mnk[3 * idx[i]], N = (double)mnk[3 * idx[i] + 1], K = (double)mnk[3 * idx[i] + 2];
        bytes += N * K + M * K + 4.0 * M * N;
    }
    std::vector<std::pair<float, int64_t>> free;   // when slots are free, and how many
    for (const int t : TRY) {
        if (t >= COARSE && !finer) continue;
        const Tile &T = TILES[t];
        const int64_t slots = (int64_t)cus * T.per_cu;
        free.assign(1, {0.0f, slots});
        float end = 0.0f;
        int64_t count = 0;
        for (int i = 0; i < n; ++i) {
            const int64_t M = mnk[3 * idx[i]], N = mnk[3 * idx[i] + 1], nk = mnk[3 * idx[i] + 2] >> 7;
            int64_t tiles = ((M + T.bm - 1) / T.bm) * ((N + T.bn - 1) / T.bn);
            count += tiles;
            const float cost = PER_ROUND + (T.per_cu == 2 ? 1.0f + BESIDE : 1.0f) * alone(T, nk);
            while (tiles > 0) {   // as many tiles as slots are free first, all at once
                const size_t at = (size_t)(std::min_element(free.begin(), free.end()) - free.begin());
                const int64_t k = std::min(tiles, free[at].second);
                const float done = free[at].first + cost;
                tiles -= k;
                if (k == free[at].second) free[at].first = done;
                else {
                    free[at].second -= k;
                    free.push_back({done, k});
                }
                end = std::max(end, done);
            }
        }
        if (count > slots) end *= 1.25f;
        else if (t >= COARSE) end *= 1.15f;
        if (best < 0.0f || end < best) {
            best = end;
            *which = t;
        }
    }
    return with_memory(best, bytes);
}

template <bool DEQ>
int32_t launch_deep_batch(int which, const DeepProblem *p, int n, hipStream_t s)
{
    using namespace deep;
    if (n < 1 || n > DEEP_MAX) return MI_EINVAL;
    Batch b = {};
    for (int i = 0; i < n; ++i) b.p[i] = p[i];
    b.n = n;
    switch (which) {
    case 0: return launch_batch<Cfg<4, 4, 2, 2, 2, 5>, DEQ>(b, s);
    case 1: return launch_batch<Cfg<4, 2, 2, 2, 2, 6>, DEQ>(b, s);
    case 2: return launch_batch<Cfg<2, 2, 2, 2, 2, 5>, DEQ>(b, s);
    case 10: return launch_batch<Cfg<5, 4, 2, 2, 2, 4>, DEQ>(b, s);
    case 13: return launch_batch<Cfg<6, 4, 2, 2, 2, 4>, DEQ>(b, s);
    default: return MI_EINVAL;
    }
}
template int32_t launch_deep_batch<true>(int, const DeepProblem *, int, hipStream_t);
template int32_t launch_deep_batch<false>(int, const DeepProblem *, int, hipStream_t);

}  // namespace mi
