// Several W8A8 contractions in ONE launch, in tiles of 256 x 128: the list kernel's half-width sibling, for batches of too few
// 256 x 256 tiles to level out (gemm_list.hip decides).
//   acc[m,n] = sum_k qx[m,k] * qw[n,k],   y = ((float)acc * sx[m]) * sw[n]      (per problem of the batch)
//
// A workgroup of twelve waves per compute unit walks a list of tiles, and the K stages of all its tiles form one stream: stages
// of 128 bytes of K (48 KB) go straight to LDS through a ring of three buffers whose loads run ahead across tile boundaries, so
// that launch, first round trip and drain are paid once.  Four of the waves only load: they issue the direct-to-LDS loads, wait
// for them and say by the barrier that a stage has landed.  The other eight never wait for memory: each owns 64 x 64 results
// over the whole of K (4 x 4 matrix-instruction tiles in 64 registers; fragments of half a stage in 32 and of the other half in
// 32 more), nothing is exchanged between them, and a tile's end is a straight run of conversions and stores while the next tile's
// loads land.  One barrier a stage: it says that the next stage has landed and that everybody holds the rest of this stage in
// registers; behind it a wave requests the first half of the next stage and multiplies the second half of this one.
// A tile that would cross the edge of its matrix is moved inwards, as in gemm_list.hip.
//
// Why waves of their own.  A load of 1 KB holds the issue of the wave that makes it for as long as the path to the cache is
// busy, 16 clocks at best and 28 as measured, and the matrix instructions behind it wait: with the loads dealt to the eight
// waves, between groups of four matrix instructions, four projections with 509 rows took 129.5 us behind their quantizer, 122.5
// now, with 2048 rows (forced into these tiles) 419 and 390 for the contraction alone.  Two loading waves measured the same as four.
//
// What bounds it.  The part's power limit and the longest list: with 509 rows the units that hold a tile of K = 14336 walk 112
// stages where the mean is 96.  256 x 256 tiles move fewer bytes per result and are 1.1 times as fast where there are enough of
// them (2048 rows 353 us); 128 x 128 tiles in the form without loading waves were slower than both (509 rows 144 us).
//
// The scales of a tile come through LDS as well (in two areas by turns, 64 to a load with the tile's first stage.  The loads run
// D - 1 stages ahead: with no more than D stages a tile they could enter the tile after the next, and write its scales over those
// of the tile in work, before its end has read them.  So a tile has more stages than the ring has buffers).
#include "common.h"
#include "gemm_stream.h"
#include "lds_ops.h"

namespace mi {
namespace stream {

template <int TM_, int TN_, int WM_, int WN_, int D_, int NL_>
struct Cfg {
    static constexpr int TM = TM_, TN = TN_, WM = WM_, WN = WN_, D = D_, NL = NL_;   // a wave's tile in 16 x 16, waves, stage buffers, loading waves
    static constexpr int NW = WM * WN, BM = 16 * TM * WM, BN = 16 * TN * WN, TPB = 64 * (NW + NL);
    static constexpr int LX = BM / 8 / NL, LW = BN / 8 / NL, L = LX + LW;    // loads of a loading wave per stage (1 KB: 8 rows x 128 B)
    static constexpr int STAGE = (BM + BN) * 128, SCALES = (BM + BN) * 4, SEGS = (BM + BN) / 64;
    static constexpr int LS = (SEGS + NL - 1) / NL;                          // and of scales per tile
    static constexpr int LDS = D * STAGE + 2 * SCALES;
    static_assert(BM % 64 == 0 && BN % 64 == 0 && TN % 2 == 0 && NL % 2 == 0 && BM / 8 % NL == 0 && BN / 8 % NL == 0, "");
    static_assert(LDS <= 160 * 1024 && (D - 1) * L + 2 * LS < 63, "vmcnt counts to 63");
};

template <typename C, bool DEQ>
__global__ __launch_bounds__(C::TPB) void k_w8a8_stream(const StreamBatch bt, const v2i *__restrict__ lists, int per_wg)
{
    constexpr int TM = C::TM, TN = C::TN, D = C::D, L = C::L;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const v2i *const my = lists + (int64_t)blockIdx.x * per_wg;
    v2i e = my[0];   // {first row, first column | problem} or {-1, .}
    if (e[0] < 0) return;

    // ---- the loading waves.  The cursor stands on a stage of a tile.  Wave w fills blocks w, w + NL, ... of the activations'
    // and of the weights' part of a stage (all of w's parity, as NL is even); lane 8 * rho + c fetches chunk c ^ sigma of row rho
    if (wave >= C::NW) {
        const int w = wave - C::NW;
        const unsigned lds0 = (unsigned)(uintptr_t)(lptr_t)smem;
        const int8_t *lx = nullptr, *lw = nullptr;
        unsigned voff = 0, block = 0;
        int k = 0, nk = 0, it = 0;   // stage, stages of its tile, position in the list
        bool more = true;            // the cursor stands on a stage that exists
        auto enter = [&](const v2i &t) {
            const StreamProblem &P = bt.p[t[1] & 15];
            const int K = P.K, n0 = t[1] & ~15;
            k = 0;
            nk = K >> 7;
            lx = P.qx + (int64_t)t[0] * K;
            lw = P.qw + (int64_t)n0 * K;
            block = 8u * (unsigned)K;
            voff = (unsigned)(lane >> 3) * (unsigned)K + (unsigned)(((lane & 7) ^ (((w & 1) << 2) | (lane >> 4))) << 4);
            if constexpr (DEQ) {   // the tile's scales, 64 to a load (the last waves fetch the last 64 again)
#pragma unroll
                for (int i = 0; i < C::LS; ++i) {
                    constexpr int SX = C::BM / 64;
                    const int seg = min(w + C::NL * i, C::SEGS - 1);
                    const float *s = seg < SX ? P.sx + t[0] + seg * 64 : P.sw + n0 + (seg - SX) * 64;
                    dma4(s, (unsigned)lane * 4, lds0 + D * C::STAGE + (it & 1) * C::SCALES + seg * 256);
                }
            }
        };
        auto issue = [&](unsigned buf) {
#pragma unroll
            for (int i = 0; i < L; ++i) {
                const int b = w + C::NL * (i < C::LX ? i : i - C::LX);
                dma16(i < C::LX ? lx : lw, voff + (unsigned)k * 128u + (unsigned)b * block,
                      lds0 + buf + (i < C::LX ? 0 : C::BM * 128) + b * 1024);
            }
            if (++k == nk) {
                const v2i t = my[++it];
                if (t[0] >= 0) enter(t);
                else more = false;
            }
        };
        enter(e);
        int ahead = 0;   // stages requested
        for (; ahead < D - 1 && more; ++ahead) issue(ahead * C::STAGE);
        wait_vm<0>();
        __builtin_amdgcn_s_barrier();   // the first stage has landed
        unsigned buf = (D - 1) * C::STAGE;
        while (more) {
            issue(buf);   // into the buffer that the barrier freed
            buf = buf + C::STAGE == D * C::STAGE ? 0 : buf + C::STAGE;
            wait_vm<(D - 2) * L>();   // loads end in order: all but those of the D - 2 youngest stages, or fewer, have landed
            __builtin_amdgcn_s_barrier();
        }
        wait_vm<0>();
        for (int i = 1; i < ahead; ++i) __builtin_amdgcn_s_barrier();   // the stages that had been requested last
        return;
    }

    // ---- the multiplying waves: wave (wm, wn)
    const int wm = wave / C::WN, wn = wave % C::WN;
    const int r = lane & 15, g = lane >> 4;
    const char *x0, *x1, *w0, *w1;   // of K half 0 and 1
    {
        const int rho = r & 7, par = r >> 3, sigma = (par << 2) | (rho >> 1);
        const char *const xb = smem + wm * TM * 2048 + par * 1024, *const wb = smem + C::BM * 128 + wn * TN * 2048 + par * 1024;
        x0 = xb + ((8 * rho + (g ^ sigma)) << 4);
        x1 = xb + ((8 * rho + ((4 + g) ^ sigma)) << 4);
        w0 = wb + ((8 * rho + (g ^ sigma)) << 4);
        w1 = wb + ((8 * rho + ((4 + g) ^ sigma)) << 4);
    }
    struct Half {
        v4i x[TM], w[TN];
    };
    auto fetch = [&](Half &f, const char *xp, const char *wp, unsigned buf) {
#pragma unroll
        for (int j = 0; j < TN; ++j) f.w[j] = *reinterpret_cast<const v4i *>(wp + buf + j * 2048);
#pragma unroll
        for (int i = 0; i < TM; ++i) f.x[i] = *reinterpret_cast<const v4i *>(xp + buf + i * 2048);
    };
    v4i acc[TM * TN];
    auto clear = [&]() {
#pragma unroll
        for (int f = 0; f < TM * TN; ++f) acc[f] = (v4i){0, 0, 0, 0};
    };
    // ---- the tile in work
    int it = 0, k = 0, nk = bt.p[e[1] & 15].K >> 7;
    unsigned cur = 0;
    auto multiply = [&](const Half &f) {
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int i = 0; i < TM; ++i) acc[i * TN + j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(f.w[j], f.x[i], acc[i * TN + j], 0, 0, 0);
    };
    // the tile's results leave: two column tiles side by side trade halves between lanes r and r ^ 8, so that a store writes
    // 8 rows x 128 bytes.  false: it was the last tile
    auto finish = [&]() {
        const StreamProblem &P = bt.p[e[1] & 15];
        const int64_t N = P.N;
        const bool lo = r < 8;
        const float *const sx = reinterpret_cast<const float *>(smem + D * C::STAGE + (it & 1) * C::SCALES) + wm * TM * 16;
        const float *const sw = reinterpret_cast<const float *>(smem + D * C::STAGE + (it & 1) * C::SCALES) + C::BM + wn * TN * 16;
        char *const out = static_cast<char *>(P.out) +
                          ((e[0] + wm * TM * 16 + (r & 7)) * N + (e[1] & ~15) + wn * TN * 16 + (lo ? 0 : 16) + 4 * g) * 4;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            float sa = 1.0f, sb = 1.0f;
            if constexpr (DEQ) {
                sa = sx[i * 16 + (r & 7)];
                sb = sx[i * 16 + 8 + (r & 7)];
            }
#pragma unroll
            for (int j = 0; j < TN; j += 2) {
                const v4i t0 = acc[i * TN + j], t1 = acc[i * TN + j + 1];
                v4i va, vb;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int u0 = ror8(t0[q]), u1 = ror8(t1[q]);
                    va[q] = lo ? t0[q] : u1;
                    vb[q] = lo ? u0 : t1[q];
                }
                char *const at = out + i * 64 * N + j * 64;
                if constexpr (DEQ) {
                    const v4f s4 = *reinterpret_cast<const v4f *>(sw + j * 16 + (lo ? 0 : 16) + 4 * g);
                    v4f fa, fb;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        fa[q] = ((float)va[q] * sa) * s4[q];
                        fb[q] = ((float)vb[q] * sb) * s4[q];
                    }
                    __builtin_nontemporal_store(fa, reinterpret_cast<v4f *>(at));
                    __builtin_nontemporal_store(fb, reinterpret_cast<v4f *>(at + 32 * N));
                } else {
                    __builtin_nontemporal_store(va, reinterpret_cast<v4i *>(at));
                    __builtin_nontemporal_store(vb, reinterpret_cast<v4i *>(at + 32 * N));
                }
            }
        }
        e = my[++it];
        if (e[0] < 0) return false;
        nk = bt.p[e[1] & 15].K >> 7;
        k = 0;
        clear();
        return true;
    };

    Half f0, f1;
    clear();
    bool last = my[1][0] < 0;
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    fetch(f0, x0, w0, 0);
    for (;;) {
        fetch(f1, x1, w1, cur);
        __builtin_amdgcn_sched_barrier(0);
        multiply(f0);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0), as an instruction that the compiler's own counting sees: the stage is in registers
        const bool end = ++k == nk;
        cur = cur + C::STAGE == D * C::STAGE ? 0 : cur + C::STAGE;
        if (!(end && last)) {
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            fetch(f0, x0, w0, cur);
        }
        __builtin_amdgcn_sched_barrier(0);
        multiply(f1);
        __builtin_amdgcn_sched_barrier(0);
        if (end) {
            if (!finish()) break;
            last = my[it + 1][0] < 0;
        }
    }
}

}  // namespace stream

template <bool DEQ>
int32_t launch_stream(const StreamBatch &b, const v2i *lists, int grid, int per_wg, hipStream_t s)
{
    using C = stream::Cfg<4, 4, 4, 2, 3, 4>;
    static_assert(C::BM == 256 && C::BN == STREAM_BN, "the tiles that the lists are made of");
    static_assert(STREAM_MIN_K / 128 > C::D, "the scales of a tile are read before those of the tile after the next arrive");
    MI_LDS_OPT_IN((&stream::k_w8a8_stream<C, DEQ>), C::LDS);
    launch_kernel((stream::k_w8a8_stream<C, DEQ>), dim3((unsigned)grid), dim3(C::TPB), C::LDS, s, b, lists, per_wg);
    return launch_status();
}
template int32_t launch_stream<true>(const StreamBatch &, const v2i *, int, int, hipStream_t);
template int32_t launch_stream<false>(const StreamBatch &, const v2i *, int, int, hipStream_t);

}  // namespace mi
