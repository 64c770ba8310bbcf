// Several W8A8 contractions in ONE launch, in tiles of 256 x 128: the list kernel's half-width sibling, for batches of too few
// 256 x 256 tiles to level out (gemm_list.hip decides).
//   acc[m,n] = sum_k qx[m,k] * qw[n,k],   y = ((float)acc * sx[m]) * sw[n]      (per problem of the batch)
//
// A workgroup of eight waves per compute unit walks a list of tiles, and the K stages of all its tiles form one stream: stages
// of 128 bytes of K (48 KB) go straight to LDS through a ring of three buffers whose loads run ahead across tile boundaries, so
// that launch, first round trip and drain are paid once.  A wave owns 64 x 64 results over the whole of K (4 x 4 matrix-instruction
// tiles in 64 registers; two sets of fragments of a whole stage in 128): nothing is exchanged between waves, and a tile's end is
// a straight run of conversions and stores while the next tile's loads land and its first fragments are in registers.  One
// barrier a stage: it says that the next stage has landed and that everybody holds this stage's fragments in registers; behind
// it a wave requests the next stage's fragments and the loads into the buffer just freed, two fragments and at most one load
// between groups of four matrix instructions (in front of all 32 of them the stage took 0.96 instead of 0.84 us).
// A tile that would cross the edge of its matrix is moved inwards, as in gemm_list.hip.
//
// What bounds it.  A stage takes 0.84 us on a full chip (2.55 POP/s), 0.71 without its loads, 0.63 with neither loads nor
// fragment reads on an otherwise idle chip (variants of the kernel that are not kept), for 0.43 of matrix instructions at 2.4 GHz:
// the loads' share of the issue slots and the part's power limit.  A whole launch of the four projections with 509 rows keeps the
// matrix pipe busy 43 % of its clocks at 2.06 GHz and fetches 252 MB for 215 MB of operands.  A tile's end costs about ten stages when every unit stores its 128 KB at once.  256 x 256 tiles move
// fewer bytes per result and are 1.2 times as fast where there are enough of them; 128 x 128 tiles in this form were slower
// than both (four projections with 509 rows 144 us, this kernel 115, 256 x 256 and small tiles in two launches 135).
//
// The scales of a tile come through LDS as well (a load of 64 for each wave with the tile's first stage, in two areas by turns.
// The loads run D stages ahead: with no more than D stages a tile they would enter the tile after the next, and write its
// scales over those of the tile in work, before its end has read them.  So a tile has more stages than the ring has buffers).
#include "common.h"
#include "gemm_stream.h"
#include "lds_ops.h"

namespace mi {
namespace stream {

template <int TM_, int TN_, int WM_, int WN_, int D_>
struct Cfg {
    static constexpr int TM = TM_, TN = TN_, WM = WM_, WN = WN_, D = D_;   // a wave's tile in 16 x 16, waves, stage buffers
    static constexpr int NW = WM * WN, BM = 16 * TM * WM, BN = 16 * TN * WN;
    static constexpr int LX = BM / 8 / NW, LW = BN / 8 / NW, L = LX + LW;    // loads of a wave per stage (1 KB: 8 rows x 128 B)
    static constexpr int STAGE = L * NW * 1024, SCALES = (BM + BN) * 4;
    static constexpr int LDS = D * STAGE + 2 * SCALES;
    static constexpr int NST = TM * TN;                                       // store instructions of a wave per tile
    static_assert(NW == 8 && BM % 64 == 0 && BN % 64 == 0 && TN % 2 == 0 && LDS <= 160 * 1024, "");
    static_assert((D - 2) * L + NST < 60 && D * L < 60, "vmcnt counts to 63");
};

template <typename C, bool DEQ>
__global__ __launch_bounds__(512, 2) void k_w8a8_stream(const StreamBatch bt, const v2i *__restrict__ lists, int per_wg)
{
    constexpr int TM = C::TM, TN = C::TN, D = C::D, L = C::L;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const v2i *const my = lists + (int64_t)blockIdx.x * per_wg;
    v2i e = my[0];   // {first row, first column | problem} or {-1, .}
    if (e[0] < 0) return;

    // ---- load side: the cursor stands on a stage of a tile.  Load i of wave w fills block w + 8 i of a stage; lane
    // 8 * rho + c fetches chunk c ^ sigma of row rho of the block
    const unsigned lds0 = (unsigned)(uintptr_t)(lptr_t)smem;
    const int8_t *lx = nullptr, *lw = nullptr;
    unsigned lvoff = 0, lstep = 0;
    int lk = 0, lnk = 0, lit = 0;   // stage, stages of its tile, position in the list
    bool more = true;               // the cursor stands on a stage that exists
    auto enter = [&](const v2i &t) {
        const StreamProblem &P = bt.p[t[1] & 15];
        const int K = P.K, n0 = t[1] & ~15;
        lk = 0;
        lnk = K >> 7;
        lx = P.qx + (int64_t)t[0] * K;
        lw = P.qw + (int64_t)n0 * K;
        lstep = 64u * (unsigned)K;
        const int row = wave * 8 + (lane >> 3);
        lvoff = (unsigned)row * (unsigned)K + (unsigned)(((lane & 7) ^ (((wave & 1) << 2) | (lane >> 4))) << 4);
        if constexpr (DEQ) {   // the tile's scales, 64 to a wave (the last waves fetch the last 64 again)
            constexpr int SX = C::BM / 64, ALL = (C::BM + C::BN) / 64;
            const int seg = wave < ALL ? wave : ALL - 1;
            const float *s = seg < SX ? P.sx + t[0] + seg * 64 : P.sw + n0 + (seg - SX) * 64;
            dma4(s, (unsigned)lane * 4, lds0 + D * C::STAGE + (lit & 1) * C::SCALES + seg * 256);
        }
    };
    auto issue_one = [&](int i, unsigned buf) {   // load i of the cursor's stage
        const unsigned by = (unsigned)lk * 128u + (unsigned)(i < C::LX ? i : i - C::LX) * lstep;
        dma16(i < C::LX ? lx : lw, lvoff + by, lds0 + buf + wave * 1024 + i * 8192);
    };
    auto advance = [&]() {
        if (++lk == lnk) {
            const v2i t = my[++lit];
            if (t[0] >= 0) enter(t);
            else more = false;
        }
    };
    auto issue = [&](unsigned buf) {
        if (!more) return;
#pragma unroll
        for (int i = 0; i < L; ++i) issue_one(i, buf);
        advance();
    };

    // ---- read side: wave (wm, wn)
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
    struct Frags {
        v4i x[2][TM], w[2][TN];
    };
    auto fetch_one = [&](Frags &f, unsigned buf, int n) {   // fragment n of 2 (TM + TN)
        const int h = n / (TM + TN), m = n % (TM + TN);
        if (m < TN) f.w[h][m] = *reinterpret_cast<const v4i *>((h ? w1 : w0) + buf + m * 2048);
        else f.x[h][m - TN] = *reinterpret_cast<const v4i *>((h ? x1 : x0) + buf + (m - TN) * 2048);
    };
    v4i acc[TM * TN];
    auto clear = [&]() {
#pragma unroll
        for (int f = 0; f < TM * TN; ++f) acc[f] = (v4i){0, 0, 0, 0};
    };

    // ---- the tile in work
    int it = 0, k = 0, nk = bt.p[e[1] & 15].K >> 7;
    int since = D;   // stages since the last tile's stores
    unsigned cur = 0;
    auto stage = [&](Frags &now, Frags &next) {
        const unsigned nxt = cur + C::STAGE == D * C::STAGE ? 0 : cur + C::STAGE;
        // this stage's fragments are in registers and the next stage has landed; behind the barrier both hold for all waves.
        // Memory operations end in order; behind the next stage's loads came those of D - 2 more and, for D - 1 stages, the
        // stores of the tile before
        __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0), as an instruction that the compiler's own counting sees
        if (!more) wait_vm<0>();
        else if (since < D - 1) wait_vm<(D - 2) * L + C::NST>();
        else wait_vm<(D - 2) * L>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        ++since;
        // the next stage's fragments (behind the last stage: what an older stage left, never used) and the loads of stage + D,
        // between the matrix instructions
        constexpr int GROUPS = 2 * TN, READS = 2 * (TM + TN);
        const bool ld = more;
#pragma unroll
        for (int n = 0; n < GROUPS; ++n) {
#pragma unroll
            for (int f = READS * n / GROUPS; f < READS * (n + 1) / GROUPS; ++f) fetch_one(next, nxt, f);
#pragma unroll
            for (int l = L * n / GROUPS; l < L * (n + 1) / GROUPS; ++l)
                if (ld) issue_one(l, cur);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < TM; ++i)
                acc[i * TN + n % TN] = __builtin_amdgcn_mfma_i32_16x16x64_i8(now.w[n / TN][n % TN], now.x[n / TN][i],
                                                                             acc[i * TN + n % TN], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (ld) advance();
        cur = nxt;
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
        since = 0;
        clear();
        return true;
    };

    enter(e);
#pragma unroll
    for (int s = 0; s < D; ++s) issue(s * C::STAGE);
    if (more) wait_vm<(D - 1) * L>();   // the first stage has landed
    else wait_vm<0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    Frags fa, fb;
#pragma unroll
    for (int n = 0; n < 2 * (TM + TN); ++n) fetch_one(fa, 0, n);
    clear();
    for (;;) {
        stage(fa, fb);
        if (++k == nk && !finish()) break;
        stage(fb, fa);
        if (++k == nk && !finish()) break;
    }
}

}  // namespace stream

template <bool DEQ>
int32_t launch_stream(const StreamBatch &b, const v2i *lists, int grid, int per_wg, hipStream_t s)
{
    using C = stream::Cfg<4, 4, 4, 2, 3>;
    static_assert(C::BM == 256 && C::BN == STREAM_BN, "the tiles that the lists are made of");
    static_assert(STREAM_MIN_K / 128 > C::D, "the scales of a tile are read before those of the tile after the next arrive");
    MI_LDS_OPT_IN((&stream::k_w8a8_stream<C, DEQ>), C::LDS);
    launch_kernel((stream::k_w8a8_stream<C, DEQ>), dim3((unsigned)grid), dim3(512), C::LDS, s, b, lists, per_wg);
    return launch_status();
}
template int32_t launch_stream<true>(const StreamBatch &, const v2i *, int, int, hipStream_t);
template int32_t launch_stream<false>(const StreamBatch &, const v2i *, int, int, hipStream_t);

}  // namespace mi
