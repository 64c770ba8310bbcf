// Grouped-query decode attention over an int8 KV cache stored in the layouts the int8 matrix instruction loads
// straight from memory, 1 KB contiguous per wave instruction:
//   kt int8 [B, Hkv, T_cap/16, 8, 16, 16]  (tile of 16 tokens; byte (c, t % 16, e) = code 16*c + e of token t)
//   vt int8 [B, Hkv, T_cap/64, 8, 4, 16, 16]  (block of 64 tokens, transposed and cut into 16 x 16 pieces;
//                                           byte (d / 16, (t % 64) / 16, d % 16, t % 16) = code d of token t)
// A key load in operand layout (lane l: token l%16, 16-byte chunk l/16) is then lanes 0..63 reading consecutive
// 16-byte pieces, where the row-major cache [T, 128] makes the same load touch 16 lines of 128 bytes by halves.
// With tokens contiguous per head-dim row, a 16-byte load is 16 tokens of one output column, which is what the
// int8 matrix instruction wants for the contraction over tokens.  Both products of the attention then run on
// v_mfma_i32_16x16x64_i8 and no V byte is ever converted on the vector pipe:
//
//   scores   dots[t, h] = sum_d kq[t, d] * qq[h, d]          A = 16 tokens x 64 d, B = 64 d x 16 (G heads used)
//   P.V      o[h, d]    = sum_t p[t, h] * vs[t] * vq[t, d]   A = 16 rows x 64 tokens, B = a vt piece (64 t x 16 d)
//
// For the second product the fp32 weights a[t, h] = exp2(s[t, h] - m[h]) * vs[t] are written as fixed-point
// numbers of 28 bits relative to the largest V scale of the workgroup's span, in workgroups of eight waves of the 64-token
// block (rounded to nearest: a token whose V
// scale is 1/r of that largest one keeps 28 - log2(r) bits of its weight, more than fp32's 24 while r < 16) and
// cut into four 7-bit digits; digit k of head h is row 4*k + h of A, so that ONE instruction multiplies all four
// digits of the four heads with the block, and the four int32 partial sums are recombined in fp32 when the wave is
// done (with eight waves: when the block is).  Inside a wave, or a block, the sums are exact integers (any order), across them fp32.
//
// A workgroup of four waves (eight where it sees a whole sequence of 257 to 1024 tokens) owns one span of 64-token blocks of one
// (batch, kv head) row; wave w takes blocks w, w + 4 (w + 8), ... of it.  Pass 1 streams the wave's key blocks (8 loads of 1 KB each) and leaves the scores in LDS;
// pass 2 streams the value blocks.  All loads run through one ring of register slots that is refilled slot by slot,
// keys first, values behind them, so that the same number of bytes stays in flight from the first instruction to
// the last.  The per-token scales of the span are staged in LDS once, up front.
//
// The partial results have the layout the merge kernels of attention.hip take.
//
// Bound: HBM (the K and V codes, 2 * B * Hkv * T * 128 bytes, + 8 bytes of scales per token-head).
#include <algorithm>

#include "fwht_core.h"

namespace mi {
bool row_takes(int64_t N, int64_t K);   // gemv.hip
bool merged_takes(int splits, int64_t N, int64_t K);
namespace attn {
int max_splits(int64_t B, int64_t Hkv, int64_t T);   // the row-major layout's plan: the largest split count for any length up to T
int merge_batches(int splits, int64_t rows, bool quant);
int32_t launch_merge(const float *part_o, const float *part_ml, float *o, int8_t *oq, float *oscale, int64_t B,
                     int64_t Hq, int64_t Hkv, int splits, int out_rotated, hipStream_t s);
}
namespace avt {

constexpr int D = 128;
constexpr int SROW = 64 + 16;                // floats per (head, block) score row: rows 64 bytes apart modulo the
                                             // 256 bytes an LDS cycle serves, so that the 16 lanes of a group hit
                                             // 16 distinct 16-byte slots in both passes
constexpr float FIX_ONE = 268435200.0f;      // 2^28 - 256: the fixed-point image of the largest weight

struct Params {
    const float *q;
    const int8_t *kq;
    const float *ks;
    const int8_t *vt;
    const float *vs;
    float *part_o;    // [B*Hkv, splits, 4, 128]
    float *part_ml;   // [B*Hkv, splits, 2, 4]   (max in log2 units, sum)
    int Hq, Hkv, G, T;
    int Tstride;              // tokens between consecutive (batch, kv head) rows of the cache, a multiple of 64
    const int32_t *seq_len;   // per-sequence token counts [B] (device), or null: every sequence holds T tokens
    int blocks_per_split;     // 64-token blocks per workgroup, <= NW * NT
    float score_scale;        // log2(e) / sqrt(D)
    float *o;                 // DIRECT kernels: the output rows [B, Hq, 128]
    int out_rotated;
    // paged cache: kq / vt are pools of 8 KB blocks [page][kv head], ks / vs pools of 64 scales [page][kv head];
    // 64-token block i of sequence b lives in page block_table[b * max_pages + i].  Null: the dense layout.
    const int32_t *block_table;
    int max_pages;
    // gate outputs (null in production): the int8 query codes [B, Hq, 128], their scales [B, Hq] and the raw int32
    // dots [B, Hq, T] this kernel works from
    int8_t *dbg_qq;
    float *dbg_sq;
    int32_t *dbg_dots;
};

// APPEND kernels: fused QKV rows [Hq | Hkv | Hkv] x 128 in place of q, the rotary tables, and the position that each
// sequence's new token takes in the cache; q receives the rotated query rows.  A type of its own: with these in Params the
// kernels that append nothing took up to 5 % longer (14 sequences of 475 tokens, 4 heads: 8.13 -> 8.53 us).
struct StepParams : Params {
    int splits;               // workgroups per row (gridDim.x would be one more cache line of arguments)
    const float *qkv;
    int64_t qkv_stride;
    const float *cs, *sn;
    const int32_t *pos;
};

// Rotary embedding of the eight elements 4 j .. and 64 + 4 j .. of a head (the arithmetic of k_rope_kv_append, layer_ops.hip)
__device__ __forceinline__ void rope8(float (&v)[8], const float4 &c4, const float4 &s4)
{
    const float c[4] = {c4.x, c4.y, c4.z, c4.w}, s[4] = {s4.x, s4.y, s4.z, s4.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float a = v[e], bb = v[e + 4];
        v[e] = a * c[e] - bb * s[e];
        v[e + 4] = bb * c[e] + a * s[e];
    }
}

// Codes 4 j .. (c0) and 64 + 4 j .. (c1) of a head of token tp to their place; blk0: first token of its 64-token block
__device__ __forceinline__ void store_token(bool is_v, int j, int tp, int64_t blk0, uint32_t c0, uint32_t c1, int8_t *kq,
                                            int8_t *vt)
{
    if (!is_v) {
        // codes 4j .. 4j+3: chunk j/4, bytes 4*(j%4) .. of token tp % 16 in tile tp / 16; codes 64 + 4j ..: chunk 4 + j/4
        int8_t *q = kq + (blk0 + (tp & 48)) * D + (j >> 2) * 256 + (tp & 15) * 16 + 4 * (j & 3);
        *reinterpret_cast<uint32_t *>(q) = c0;
        *reinterpret_cast<uint32_t *>(q + 1024) = c1;
    } else {
        // code d of token tp: block tp / 64, piece d / 16, token chunk (tp % 64) / 16, row d % 16, byte tp % 16
        int8_t *blk = vt + blk0 * D + (j >> 2) * 1024 + ((tp & 63) >> 4) * 256 + 4 * (j & 3) * 16 + (tp & 15);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            blk[e * 16] = (int8_t)(c0 >> (8 * e));
            blk[4096 + e * 16] = (int8_t)(c1 >> (8 * e));
        }
    }
}

// NW: waves per workgroup; NT: blocks per wave; RING: 1 KB loads a wave keeps in flight (8 or 16).
// DIRECT: the workgroup covers the whole sequence (one split): it normalizes and writes the output rows itself and
// no partial result leaves the chip.
// APPEND: the decode step's rotary embedding and cache append happen here instead of in a launch of their own (dense
// layout).  Every wave rotates its own copy of the query rows; the one wave in the grid whose block holds the new token
// (the last split's first wave if no block does) quantizes the key and value heads, stores them, and only then requests
// its blocks: nobody else reads that token.  The new scales meet the loaded ones in LDS.  A launch of its own takes 4 to 5
// us of latency for a few KB; here it is one more memory round trip in a few workgroups.  Decode steps, us with two
// launches -> one: 16 sequences of 4096 tokens, four layers 402 -> 392; one of 1531, four layers 300 -> 287; 16 of 1024
// with experts, two layers 286 -> 280.
template <int NW, int NTM, int RING, bool DIRECT, bool APPEND>
__global__ __launch_bounds__(64 * NW, NW > 4 ? 2 : APPEND ? 1 : NTM > 1 ? 3 : 4) void k_gqa_tiled_split(std::conditional_t<APPEND, StepParams, Params> p)
{
    constexpr int SPAN = NW * NTM * 64;                   // tokens a workgroup can cover
    // What the weights' fixed point is relative to: the largest V scale of the span, or, in the span of eight waves, that of each block,
    // whose sums become fp32 by themselves.  That span is as long as the two to four of four waves that it stands for: relative to its
    // largest scale a token keeps fewer bits than there.  Relative 2-norm error against 64-bit sums, 11 shapes of 270 to 1024 tokens, spans
    // of four waves and a merge / one scale for eight waves / one a block: scales alike 2.68 / 2.66 / 2.66e-7, spread over a factor of
    // 4096 2.69 / 2.68 / 2.68e-7, one token's 256 times the others' 12.0 / 15.0 / 5.4e-7.
    constexpr bool BY_BLOCK = NW > 4;
    static_assert(!(BY_BLOCK && APPEND), "a new token's scale counts for the span");
    constexpr int SC_BYTES = NW * NTM * 4 * SROW * 4;     // scores [wave][block][head][SROW]
    constexpr int SCALE_BYTES = 2 * SPAN * 4;             // ks, vs of the span
    constexpr int RROW = D + 16;                          // so that the four heads of a store lie in different banks
    constexpr int RED_BYTES = NW * 4 * RROW * 4;          // [wave][head][RROW] fp32, reuses the space above
    constexpr int UNION = (SC_BYTES + SCALE_BYTES > RED_BYTES) ? SC_BYTES + SCALE_BYTES : RED_BYTES;
    static_assert(SPAN <= 4 * 64 * NW, "one float4 of each scale array per thread");
    __shared__ __attribute__((aligned(16))) char s_mem[UNION];
    __shared__ __attribute__((aligned(16))) int8_t s_q[NW][4][D];
    __shared__ __attribute__((aligned(16))) float s_out[4][D];
    __shared__ float s_sq[NW][4], s_vmax[BY_BLOCK ? NW * NTM : NW];
    __shared__ __attribute__((aligned(16))) float s_m[4][NW], s_l[4][NW];   // by head and wave
    float *s_sc = reinterpret_cast<float *>(s_mem);
    float *s_ks = reinterpret_cast<float *>(s_mem + SC_BYTES);
    float *s_vs = s_ks + SPAN;
    float *s_red = reinterpret_cast<float *>(s_mem);

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int split = blockIdx.x, bkv = blockIdx.y;
    const int b = bkv / p.Hkv, kvh = bkv % p.Hkv;
    const int G = p.G;
    int splits;
    if constexpr (APPEND) splits = p.splits;
    else splits = gridDim.x;
    const int64_t pbase = (int64_t)bkv * splits + split;
    const bool paged = p.block_table;

    int T = p.T;
    if (p.seq_len) T = min(max(__builtin_amdgcn_readfirstlane(p.seq_len[b]), 0), p.T);
    const int blk_lo = split * p.blocks_per_split;
    const int t_lo = blk_lo * 64;
    int tp = -1;              // the new token's position, if it has one in the cache
    bool owner = false;       // this wave appends it
    float new_ks = 0.0f, new_vs = 0.0f;
    if constexpr (APPEND) {
        tp = __builtin_amdgcn_readfirstlane(p.pos[b]);
        if (tp < 0 || tp >= p.Tstride) tp = -1;
        const int at = (tp >> 6) - blk_lo;
        const bool last = split == splits - 1;
        if (tp >= 0 && at >= 0 && (at < p.blocks_per_split || last)) owner = wave == (at < p.blocks_per_split ? at % NW : 0);
        if (owner) {
            const int j = lane & 15;
            const bool is_v = (lane >> 4) & 1;   // lanes 0 - 15: the key head, 16 - 31: the value head (and both again)
            const float *src = p.qkv + b * p.qkv_stride + (int64_t)(p.Hq + (is_v ? p.Hkv : 0) + kvh) * D + 4 * j;
            const float4 lo = *reinterpret_cast<const float4 *>(src), hi = *reinterpret_cast<const float4 *>(src + D / 2);
            float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
            if (!is_v)
                rope8(v, *reinterpret_cast<const float4 *>(p.cs + (int64_t)tp * (D / 2) + 4 * j),
                      *reinterpret_cast<const float4 *>(p.sn + (int64_t)tp * (D / 2) + 4 * j));
            fwht_codes<D>(v, j);
            const float a = max_lanes<16>(abs8(v));
            const float sc = (a == 0.0f) ? 1.0f : a / 127.0f;
            const float inv = (a == 0.0f) ? 0.0f : 127.0f / a;
            const int64_t blk0 = (int64_t)bkv * p.Tstride + (tp & ~63);
            if (lane < 32) {
                store_token(is_v, j, tp, blk0, quant4(v[0], v[1], v[2], v[3], inv), quant4(v[4], v[5], v[6], v[7], inv),
                            const_cast<int8_t *>(p.kq), const_cast<int8_t *>(p.vt));
                if (j == 0) const_cast<float *>(is_v ? p.vs : p.ks)[blk0 + (tp & 63)] = sc;
            }
            new_ks = __shfl(sc, 0, 64);
            new_vs = __shfl(sc, 16, 64);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // stored before the wave's blocks are requested
        }
    }
    if (t_lo >= T) {
        if constexpr (APPEND) {
            if (split == 0 && tp >= 0) {   // nothing to attend to; the query rows are rotated all the same
                const int hr = tid >> 4, j = tid & 15;
                if (hr < G) {
                    const int64_t row = (int64_t)(kvh * G + hr) * D + 4 * j;
                    const float *src = p.qkv + b * p.qkv_stride + row;
                    const float4 lo = *reinterpret_cast<const float4 *>(src), hi = *reinterpret_cast<const float4 *>(src + D / 2);
                    float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
                    rope8(v, *reinterpret_cast<const float4 *>(p.cs + (int64_t)tp * (D / 2) + 4 * j),
                          *reinterpret_cast<const float4 *>(p.sn + (int64_t)tp * (D / 2) + 4 * j));
                    float *dst = const_cast<float *>(p.q) + (int64_t)b * p.Hq * D + row;
                    *reinterpret_cast<float4 *>(dst) = make_float4(v[0], v[1], v[2], v[3]);
                    *reinterpret_cast<float4 *>(dst + D / 2) = make_float4(v[4], v[5], v[6], v[7]);
                }
            }
        }
        if constexpr (DIRECT) {
            // a sequence of length 0: a row of zeros
            for (int o = tid; o < G * D; o += 64 * NW) p.o[((int64_t)b * p.Hq + kvh * G) * D + o] = 0.0f;
        } else {
            // this split lies past the end of the sequence: an empty partial (weight 0 in the merge)
            for (int o = tid; o < 4 * D; o += 64 * NW) p.part_o[pbase * 4 * D + o] = 0.0f;
            if (tid < 4) {
                p.part_ml[pbase * 8 + tid] = -INFINITY;
                p.part_ml[pbase * 8 + 4 + tid] = 0.0f;
            }
        }
        return;
    }
    const int t_end = min((blk_lo + p.blocks_per_split) * 64, T);   // first token this workgroup does not own
    const int nblk_row = p.Tstride >> 6;                            // blocks per cache row

    // ---- loads, in the order they are needed: the span's scales, the query rows, the pages of the wave's blocks, then the ring
    const int last_blk = (T - 1) >> 6;   // the last block that holds a token of this sequence
    const int sidx = 4 * tid;   // one float4 of each scale array per thread
    float4 ks4 = make_float4(0.f, 0.f, 0.f, 0.f), vs4 = ks4;
    if (sidx < SPAN) {
        if (paged) {
            // four consecutive tokens lie in one page; blocks past the sequence's last one (their table entries may
            // hold anything) fall back on it, and their tokens are masked like any token past the end
            const int tb = min((t_lo + sidx) >> 6, last_blk);
            const int64_t of = p.block_table[(int64_t)b * p.max_pages + tb];
            const int64_t at = (of * p.Hkv + kvh) * 64 + ((t_lo + sidx) & 63);
            ks4 = *reinterpret_cast<const float4 *>(p.ks + at);
            vs4 = *reinterpret_cast<const float4 *>(p.vs + at);
        } else {
            const int tk = min(t_lo + sidx, p.Tstride - 4);   // the row's own memory; tokens past the end are masked
            ks4 = *reinterpret_cast<const float4 *>(p.ks + (int64_t)bkv * p.Tstride + tk);
            vs4 = *reinterpret_cast<const float4 *>(p.vs + (int64_t)bkv * p.Tstride + tk);
        }
    }
    const int hr = lane >> 4, jj = lane & 15;
    const int head = kvh * G + min(hr, G - 1);
    const float *qr = p.q + ((int64_t)b * p.Hq + head) * D;
    float4 rc4 = make_float4(1.f, 1.f, 1.f, 1.f), rs4 = make_float4(0.f, 0.f, 0.f, 0.f);
    if constexpr (APPEND) {
        if (tp >= 0) {   // (a sequence without a new token attends with what q holds)
            qr = p.qkv + b * p.qkv_stride + (int64_t)head * D;
            rc4 = *reinterpret_cast<const float4 *>(p.cs + (int64_t)tp * (D / 2) + 4 * jj);
            rs4 = *reinterpret_cast<const float4 *>(p.sn + (int64_t)tp * (D / 2) + 4 * jj);
        }
    }
    const float4 qlo = *reinterpret_cast<const float4 *>(qr + 4 * jj);
    const float4 qhi = *reinterpret_cast<const float4 *>(qr + 64 + 4 * jj);
    // One look-up per block, all of them scalar and requested at once.  (Looked up where a block's address is formed, inside the
    // branches below, they became vector loads that each waited for everything in front of them: 8 sequences of 2048 tokens 13.6
    // instead of 13.1 us, 16 of 4096 30.6 instead of 29.6.  In front of the scales: 4 % slower with one block a wave.)
    int page[NTM] = {};
    if (paged) {
        const auto *table = (const __attribute__((address_space(4))) int32_t *)(p.block_table + (int64_t)b * p.max_pages);
#pragma unroll
        for (int j = 0; j < NTM; ++j) page[j] = table[min(blk_lo + NW * j + wave, last_blk)];
    }

    // The blocks that there are, NT to a wave: a span that ends with a short sequence is streamed as the shorter one that it is
    // (16 sequences of 1024 to 4096 tokens 23.7 -> 22.3 us, 32 of 512 to 2048 25.9 -> 23.4).  The kernel that appends knows
    // four and two blocks only, and no bound on its registers: with all four lengths under one its full spans took 0.3 us more
    // (16 sequences of 4096 tokens, a step's attention and projection, 35.4 -> 35.7; so 35.4, of 1024 to 4096 31.3 -> 30.1).  In
    // pages a span is always streamed whole: its blocks past the end are the sequence's last one, out of a cache (16 sequences of
    // 1024 to 4096 tokens 22.5 us, cut short 23.1).
    auto stream = [&](auto BLOCKS) {
    constexpr int NT = decltype(BLOCKS)::value;
    // block j of this wave: index blk_lo + NW*j + wave (the waves stream neighbouring blocks); blocks past the
    // end of the cache row fall back on its last block and are masked like any token past the end
    const int r16 = lane & 15, c4 = lane >> 4;
    // (both layouts put lane l's 16 bytes at 16*l inside each 1 KB piece: uniform base + one per-lane offset)
    const unsigned loff = 16u * (unsigned)lane;
    const int8_t *kblk[NT], *vblk[NT];   // the wave's blocks: 8 KB each, at the same offset in both arrays
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        int64_t off;
        if (paged) {
            off = ((int64_t)page[j] * p.Hkv + kvh) * 8192;
        } else {
            off = ((int64_t)bkv * nblk_row + min(blk_lo + NW * j + wave, nblk_row - 1)) * 8192;
        }
        kblk[j] = p.kq + off;
        vblk[j] = p.vt + off;
    }

    // load unit u in [0, 16 * NT): units 0 .. 8*NT-1 are key loads (block u/8; 16 tokens u%8/2, d half u%2),
    // the rest value loads (block (u - 8*NT)/8; head-dim rows 16*(u%8) .. +15); unit u lives in slot u % RING
    v4i ring[RING];
    auto issue = [&](auto U) {
        constexpr int u = decltype(U)::value;
        if constexpr (u < 8 * NT) {
            constexpr int j = u / 8, sub = (u % 8) / 2, hf = u % 2;
            ring[u % RING] = *reinterpret_cast<const v4i *>(kblk[j] + (sub * 2048 + hf * 1024) + loff);
        } else if constexpr (u < 16 * NT) {
            constexpr int j = (u - 8 * NT) / 8, n = u % 8;
            ring[u % RING] = *reinterpret_cast<const v4i *>(vblk[j] + n * 1024 + loff);
        }
    };
    __builtin_amdgcn_sched_barrier(0);
    static_for<RING>([&](auto U) { issue(U); });
    __builtin_amdgcn_sched_barrier(0);

    // ---- scales of the span -> LDS, and the largest V scale among the live tokens
    {
        const float v[4] = {vs4.x, vs4.y, vs4.z, vs4.w};
        float vm = 0.0f;
#pragma unroll
        for (int e = 0; e < 4; ++e) vm = fmaxf(vm, (t_lo + sidx + e < t_end && (!APPEND || t_lo + sidx + e != tp)) ? v[e] : 0.0f);
        vm = max_lanes<BY_BLOCK ? 16 : 64>(vm);   // (16 lanes hold a block's scales)
        if (APPEND && owner && tp < t_end) vm = fmaxf(vm, new_vs);
        if (sidx < SPAN) {
            *reinterpret_cast<float4 *>(s_ks + sidx) = ks4;
            *reinterpret_cast<float4 *>(s_vs + sidx) = vs4;
            if (BY_BLOCK && (tid & 15) == 0) s_vmax[tid >> 4] = vm;
        }
        if (!BY_BLOCK && lane == 0) s_vmax[wave] = vm;
    }
    // ---- query heads of this group: every wave rotates and quantizes them for itself
    {
        float v[8] = {qlo.x, qlo.y, qlo.z, qlo.w, qhi.x, qhi.y, qhi.z, qhi.w};
        if constexpr (APPEND) {
            if (tp >= 0) {
                rope8(v, rc4, rs4);
                if (split == 0 && wave == 0 && hr < G) {
                    float *dst = const_cast<float *>(p.q) + ((int64_t)b * p.Hq + head) * D + 4 * jj;
                    *reinterpret_cast<float4 *>(dst) = make_float4(v[0], v[1], v[2], v[3]);
                    *reinterpret_cast<float4 *>(dst + D / 2) = make_float4(v[4], v[5], v[6], v[7]);
                }
            }
        }
        fwht_codes<D>(v, jj);
        const float a = max_lanes<16>(abs8(v));
        const float sc = (a == 0.0f) ? 1.0f : a / 127.0f;
        const float inv = (a == 0.0f) ? 0.0f : 127.0f / a;
        const uint32_t c0 = quant4(v[0], v[1], v[2], v[3], inv), c1 = quant4(v[4], v[5], v[6], v[7], inv);
        *reinterpret_cast<uint32_t *>(&s_q[wave][hr][4 * jj]) = c0;
        *reinterpret_cast<uint32_t *>(&s_q[wave][hr][64 + 4 * jj]) = c1;
        if (jj == 0) s_sq[wave][hr] = sc;
        if (p.dbg_qq && split == 0 && wave == 0 && hr < G) {
            int8_t *dq = p.dbg_qq + ((int64_t)b * p.Hq + head) * D;
            *reinterpret_cast<uint32_t *>(dq + 4 * jj) = c0;
            *reinterpret_cast<uint32_t *>(dq + 64 + 4 * jj) = c1;
            if (jj == 0) p.dbg_sq[(int64_t)b * p.Hq + head] = sc;
        }
    }
    // LDS only: the ring's loads stay in flight across this barrier
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (APPEND && owner && tp < t_end && lane == 0) {   // scales of the wave's own block: no one else reads them
        s_ks[tp - t_lo] = new_ks;
        s_vs[tp - t_lo] = new_vs;
    }
    float vmax = s_vmax[BY_BLOCK ? wave : 0];
#pragma unroll
    for (int w = 1; w < (BY_BLOCK ? 1 : NW); ++w) vmax = fmaxf(vmax, s_vmax[w]);
    float fix = vmax > 0.0f ? FIX_ONE / vmax : 0.0f;   // weight -> fixed point
    // MFMA operand B of the score product: column l%16 = query head (columns >= G are zero), 16-byte chunk l/16
    v4i qb0 = {0, 0, 0, 0}, qb1 = {0, 0, 0, 0};
    if (r16 < G) {
        qb0 = *reinterpret_cast<const v4i *>(&s_q[wave][r16][16 * c4]);
        qb1 = *reinterpret_cast<const v4i *>(&s_q[wave][r16][64 + 16 * c4]);
    }
    const float cq = r16 < G ? s_sq[wave][r16] * p.score_scale : 0.0f;   // this lane's head, log2 units

    // ---- pass 1: scores.  Lane (head r16, group c4) gets tokens 16*sub + 4*c4 .. +3 of each 16-token product.
    float *sc_wave = s_sc + wave * (NT * 4 * SROW);
    float mrun = -INFINITY;
    static_for<NT>([&](auto J) {
        constexpr int j = decltype(J)::value;
        const int tok0 = (blk_lo + NW * j + wave) * 64;        // first token of the block (may lie past t_end)
        const int sbase = (NW * j + wave) * 64;                // its place in the staged scales
        static_for<4>([&](auto S) {
            constexpr int sub = decltype(S)::value;
            constexpr int u = 8 * j + 2 * sub;
            v4i dots = __builtin_amdgcn_mfma_i32_16x16x64_i8(ring[u % RING], qb0, (v4i){0, 0, 0, 0}, 0, 0, 0);
            dots = __builtin_amdgcn_mfma_i32_16x16x64_i8(ring[(u + 1) % RING], qb1, dots, 0, 0, 0);
            issue(std::integral_constant<int, u + RING>{});
            issue(std::integral_constant<int, u + 1 + RING>{});
            __builtin_amdgcn_sched_barrier(0);
            const float4 kk = *reinterpret_cast<const float4 *>(s_ks + sbase + 16 * sub + 4 * c4);
            const int tt = tok0 + 16 * sub + 4 * c4;
            if (p.dbg_dots && r16 < G) {
                int32_t *dd = p.dbg_dots + ((int64_t)b * p.Hq + kvh * G + r16) * p.T;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (tt + e < t_end) dd[tt + e] = dots[e];
            }
            float4 sc;
            sc.x = (float)dots[0] * (kk.x * cq);
            sc.y = (float)dots[1] * (kk.y * cq);
            sc.z = (float)dots[2] * (kk.z * cq);
            sc.w = (float)dots[3] * (kk.w * cq);
            if (tok0 + 64 > t_end) {   // the block holds the end of the span (uniform over the wave)
                sc.x = (tt + 0 < t_end) ? sc.x : -INFINITY;
                sc.y = (tt + 1 < t_end) ? sc.y : -INFINITY;
                sc.z = (tt + 2 < t_end) ? sc.z : -INFINITY;
                sc.w = (tt + 3 < t_end) ? sc.w : -INFINITY;
            }
            if (r16 < 4) *reinterpret_cast<float4 *>(sc_wave + (j * 4 + r16) * SROW + 16 * sub + 4 * c4) = sc;
            mrun = fmaxf(fmaxf(mrun, fmaxf(sc.x, sc.y)), fmaxf(sc.z, sc.w));
        });
    });
    // maximum per head over the wave's tokens: lanes r16, r16 + 16, r16 + 32, r16 + 48 hold the partial maxima
    const auto larger = [](float a, float b) { return fmaxf(a, b); };
    mrun = with_far_lane<32>(with_far_lane<16>(mrun, larger), larger);
    if (lane < 4) s_m[lane][wave] = mrun;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

    // ---- pass 2: P.V.  Row r16 = 4*head + digit of operand A.  The four lanes of a quad share a head: lane `dg`
    // of the quad computes the weights of tokens 16*c4 + 4*dg .. +3 of the block (one exp2 per weight and lane, not
    // four), as 28-bit fixed-point codes; every lane then takes its own 7-bit digit of all 16 codes of the quad
    // (quad broadcasts).  The softmax is taken against the wave's own maximum (a wave whose tokens are all masked
    // has maximum -inf: its weights are 0, and 0 stands in for the maximum).
    const int hh = r16 >> 2, dg = r16 & 3;
    const float m_raw = s_m[hh][wave];
    const float m_h = (m_raw == -INFINITY) ? 0.0f : m_raw;
    const unsigned sh = 21u - 7u * (unsigned)dg;
    v4i acc[8];
#pragma unroll
    for (int n = 0; n < 8; ++n) acc[n] = (v4i){0, 0, 0, 0};
    // digits -> fp32.  Lane (r16, c4) holds column d = 16*n + r16 of rows 4*c4 + i: digit i of head c4, worth
    // 2^(21 - 7*i) / fix: the four digits of a value are the four registers of one lane (low digits added first).
    float val[8];
    auto value = [&](int n) {
        const float unit = vmax > 0.0f ? vmax / FIX_ONE : 0.0f;
        float f = (float)acc[n][3] * unit;
        f += (float)acc[n][2] * (unit * 128.0f);
        f += (float)acc[n][1] * (unit * 16384.0f);
        f += (float)acc[n][0] * (unit * 2097152.0f);
        return f;
    };
    float lsum = 0.0f;
    static_for<NT>([&](auto J) {
        constexpr int j = decltype(J)::value;
        if constexpr (BY_BLOCK && j > 0) {
#pragma unroll
            for (int n = 0; n < 8; ++n) {
                val[n] = j > 1 ? val[n] + value(n) : value(n);
                acc[n] = (v4i){0, 0, 0, 0};
            }
            vmax = s_vmax[NW * j + wave];
            fix = vmax > 0.0f ? FIX_ONE / vmax : 0.0f;
        }
        const float4 s4 = *reinterpret_cast<const float4 *>(sc_wave + (j * 4 + hh) * SROW + 16 * c4 + 4 * dg);
        const float4 v4 = *reinterpret_cast<const float4 *>(s_vs + (NW * j + wave) * 64 + 16 * c4 + 4 * dg);
        const float ss[4] = {s4.x, s4.y, s4.z, s4.w}, vv[4] = {v4.x, v4.y, v4.z, v4.w};
        unsigned code[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float pe = __builtin_amdgcn_exp2f(ss[e] - m_h);       // masked token: exp2(-inf) = 0
            lsum += pe;
            const float a = (pe == 0.0f) ? 0.0f : pe * (vv[e] * fix);   // (a masked token's scale may be anything)
            code[e] = min((unsigned)(a + 0.5f), 0x0fffffffu);           // to nearest; the clamp covers a = 2^28
        }
        v4i pa;
        static_for<4>([&](auto K) {
            constexpr int k = decltype(K)::value;   // tokens 16*c4 + 4*k .. +3: the codes of quad lane k
            unsigned word = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const unsigned c = (unsigned)__builtin_amdgcn_update_dpp(0, (int)code[e], k * 0x55, 0xf, 0xf, true);
                word |= ((c >> sh) & 0x7fu) << (8 * e);
            }
            pa[k] = (int)word;
        });
        static_for<8>([&](auto N) {
            constexpr int n = decltype(N)::value;
            constexpr int u = 8 * NT + 8 * j + n;
            acc[n] = __builtin_amdgcn_mfma_i32_16x16x64_i8(pa, ring[u % RING], acc[n], 0, 0, 0);
            issue(std::integral_constant<int, u + RING>{});
        });
    });
    // the sum of the weights of head hh: over the quad, then over the four chunks c4
    lsum += xor_lane<1>(lsum);
    lsum += xor_lane<2>(lsum);
    lsum = add_lane<32>(add_lane<16>(lsum));

#pragma unroll
    for (int n = 0; n < 8; ++n) val[n] = BY_BLOCK && NT > 1 ? val[n] + value(n) : value(n);
    // ---- the waves meet.  Behind the barrier every wave's maxima are known and the space of the scores and scales may be reused:
    // a wave rescales its own sums (of head c4 in this lane) to the common maximum, and what is left is adding NW numbers
    // (rescaled by the thread that adds them: NW exponentials a thread one behind the other.  One sequence of 200, 512 tokens and
    // 4096 in six spans 4.7, 5.6, 8.0 us; so 4.5, 5.4, 7.8)
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    auto common = [&](int head) {
        float m = s_m[head][0];
#pragma unroll
        for (int w = 1; w < NW; ++w) m = fmaxf(m, s_m[head][w]);
        return m;
    };
    {
        const float own = s_m[c4][wave];
        const float f = own == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(own - common(c4));
        float *dst = s_red + (wave * 4 + c4) * RROW + r16;
#pragma unroll
        for (int n = 0; n < 8; ++n) dst[16 * n] = val[n] * f;
        if (r16 == 4 * c4) s_l[c4][wave] = lsum * f;   // (hh == c4 in that lane)
    }
    __syncthreads();
    constexpr int ADD = NW < 8 ? 256 : 512;   // threads that add
    if (NW * 64 == ADD || tid < ADD) {
#pragma unroll
        for (int o = 0; o < 4 * D; o += ADD) {
            const int d = tid & (D - 1), head = (tid + o) / D;
            float sum = 0.0f, l = 0.0f;
            if constexpr (NW == 8) {   // in pairs, and divided: with V scales alike no more error than four waves and a merge (above); one by one 1.02 of it
                float a[8], b[8];
#pragma unroll
                for (int w = 0; w < 8; ++w) a[w] = s_red[(w * 4 + head) * RROW + d], b[w] = s_l[head][w];
                sum = ((a[0] + a[1]) + (a[2] + a[3])) + ((a[4] + a[5]) + (a[6] + a[7]));
                l = ((b[0] + b[1]) + (b[2] + b[3])) + ((b[4] + b[5]) + (b[6] + b[7]));
            } else {
#pragma unroll
                for (int w = 0; w < NW; ++w) {
                    sum += s_red[(w * 4 + head) * RROW + d];
                    l += s_l[head][w];
                }
            }
            if constexpr (DIRECT) {
                s_out[head][d] = l > 0.0f ? (NW == 8 ? sum / l : sum * (1.0f / l)) : 0.0f;
            } else {
                p.part_o[(pbase * 4 + head) * D + d] = sum;
                if (d == 0) {
                    p.part_ml[pbase * 8 + head] = common(head);
                    p.part_ml[pbase * 8 + 4 + head] = l;
                }
            }
        }
    }
    if constexpr (DIRECT) {
        __syncthreads();
        if (tid < 64 && hr < G) {   // 16 lanes per head row, as the merge kernel has them
            float v[8];
            const float4 lo = *reinterpret_cast<const float4 *>(&s_out[hr][4 * jj]);
            const float4 hi = *reinterpret_cast<const float4 *>(&s_out[hr][64 + 4 * jj]);
            v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w;
            v[4] = hi.x; v[5] = hi.y; v[6] = hi.z; v[7] = hi.w;
            if (!p.out_rotated) fwht_chunk<D>(v, jj);
            float *orow = p.o + ((int64_t)b * p.Hq + kvh * G + hr) * D;
            *reinterpret_cast<float4 *>(orow + 4 * jj) = make_float4(v[0], v[1], v[2], v[3]);
            *reinterpret_cast<float4 *>(orow + 64 + 4 * jj) = make_float4(v[4], v[5], v[6], v[7]);
        }
    }
    };
    const int blocks = (t_end - t_lo + 63) >> 6;
    constexpr int FEW = APPEND && NTM == 4 ? 2 : NTM - 1;
    if (NTM == 1 || (APPEND && NTM < 4) || paged || __builtin_expect(blocks > FEW * NW, 1)) stream(std::integral_constant<int, NTM>{});
    else if (APPEND) stream(std::integral_constant<int, FEW < 1 ? 1 : FEW>{});
    else if (NTM > 3 && blocks > 2 * NW) stream(std::integral_constant<int, APPEND || NTM < 3 ? 1 : 3>{});
    else if (NTM > 2 && blocks > NW) stream(std::integral_constant<int, APPEND || NTM < 2 ? 1 : 2>{});
    else stream(std::integral_constant<int, 1>{});
}

// Row-major codes [rows, src_stride tokens, 128] -> the two tiled layouts, one workgroup per (64-token block, row,
// which): keys into 16-token tiles [8 chunks][16 tokens][16 bytes] (a straight permutation of 16-byte pieces),
// values into transposed blocks through LDS (tokens >= T inside the last block touched: 0).  Latency at a prompt's size, HBM
// at a cache's.  A thread takes two head-dim rows of 16 tokens, so that a wave reads neighbouring pairs of bytes from LDS (16
// reads without a conflict; 32 single bytes with four tokens of a bank in their way before: keys and values of 8 rows of 700
// tokens 2.8 -> 2.5 us, of 2048 tokens 3.9 -> 3.7, 16 of 4096 8.1 -> 7.4, 128 of 4096 42.0 -> 41.9, at 6.4 TB/s).
__global__ __launch_bounds__(256) void k_tiled_from_rows(const int8_t *__restrict__ kq, const int8_t *__restrict__ vq,
                                                         int8_t *__restrict__ kt, int8_t *__restrict__ vt, int T,
                                                         int64_t src_stride, int64_t dst_stride, int z0)
{
    __shared__ __attribute__((aligned(16))) int8_t s[64][D + 16];
    const int tid = threadIdx.x, blk = blockIdx.x;
    const int64_t row = blockIdx.y;
    const bool is_v = (int)blockIdx.z + z0 != 0;   // z0 = 1: values only
    const int8_t *src = (is_v ? vq : kq) + (row * src_stride + (int64_t)blk * 64) * D;
    int8_t *dst = (is_v ? vt : kt) + (row * dst_stride + (int64_t)blk * 64) * D;
    if (!is_v) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int c = tid + 256 * i, t = c >> 3, part = c & 7;   // 16-byte chunk `part` of token t
            v4i v = {0, 0, 0, 0};
            if (blk * 64 + t < T) v = *reinterpret_cast<const v4i *>(src + t * D + 16 * part);
            *reinterpret_cast<v4i *>(dst + (t >> 4) * 2048 + part * 256 + (t & 15) * 16) = v;
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int c = tid + 256 * i, t = c >> 3, part = c & 7;
        v4i v = {0, 0, 0, 0};
        if (blk * 64 + t < T) v = *reinterpret_cast<const v4i *>(src + t * D + 16 * part);
        *reinterpret_cast<v4i *>(&s[t][16 * part]) = v;
    }
    __syncthreads();
    const int d = 2 * (tid & 63), part = tid >> 6;   // tokens 16*part .. +15 of head-dim rows d and d + 1
    uint32_t w[2][4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        uint32_t x[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = *reinterpret_cast<const uint16_t *>(&s[16 * part + 4 * k + e][d]);
        const uint32_t lo = x[0] | x[1] << 16, hi = x[2] | x[3] << 16;
        w[0][k] = __builtin_amdgcn_perm(hi, lo, 0x06040200u);
        w[1][k] = __builtin_amdgcn_perm(hi, lo, 0x07050301u);
    }
    int8_t *at = dst + (d >> 4) * 1024 + part * 256 + (d & 15) * 16;
    *reinterpret_cast<uint4 *>(at) = make_uint4(w[0][0], w[0][1], w[0][2], w[0][3]);
    *reinterpret_cast<uint4 *>(at + 16) = make_uint4(w[1][0], w[1][1], w[1][2], w[1][3]);
}

// The decode step's append for this layout: rotate + quantize the new token's key and value heads exactly as
// k_kv_append does (fwht_quant.hip); the key codes go to their 128-byte line, the value codes to byte t % 64 of
// the 128 head-dim rows of block t / 64.  16 lanes per head; blockIdx.y = 0: keys, 1: values.
// ROPE: rows are fused QKV rows [Hq | Hkv | Hkv] x 128 and query / key heads first get the rotary embedding
// (the arithmetic of k_rope_kv_append, layer_ops.hip); queries leave packed in q_out.
template <bool ROPE>
__global__ __launch_bounds__(256) void k_kv_append_vt(const float *__restrict__ k_new, const float *__restrict__ v_new,
                                                      int64_t row_stride, const float *__restrict__ cs,
                                                      const float *__restrict__ sn, float *__restrict__ q_out,
                                                      int8_t *__restrict__ kq, float *__restrict__ ks,
                                                      int8_t *__restrict__ vt, float *__restrict__ vs,
                                                      const int32_t *__restrict__ pos, int B, int Hq, int Hkv, int T_cap,
                                                      const int32_t *__restrict__ block_table, int max_pages)
{
    constexpr int LPB = 16;
    const int t = threadIdx.x, j = t % LPB;
    const int heads = ROPE ? Hq + 2 * Hkv : Hkv;
    const int flat = blockIdx.x * 16 + t / LPB;
    const int b = min(flat / heads, B - 1), hd = flat % heads;
    bool is_q = false, is_v;
    int h;
    const float *src;
    if constexpr (ROPE) {
        is_q = hd < Hq;
        is_v = hd >= Hq + Hkv;
        h = is_v ? hd - Hq - Hkv : hd - Hq;
        src = k_new + (int64_t)b * row_stride + (int64_t)hd * D + 4 * j;
    } else {
        is_v = blockIdx.y != 0;
        h = hd;
        src = (is_v ? v_new : k_new) + (int64_t)b * row_stride + (int64_t)h * D + 4 * j;
    }
    // All latency: the head's row does not wait for the position, and the page is looked up while the row is on its way.  us in
    // a chain of appends of 1, 16 and 32 sequences, 8 heads, before -> after: 2.9 -> 2.5, 3.6 -> 3.1, 3.7 -> 3.3 (row-major, fwht_quant.hip:
    // 2.4 -> 2.0, 2.6 -> 2.2, 2.65 -> 2.2), dense and in pages alike; of 24 with the attention behind it 27.1 -> 26.4.
    const float4 lo = *reinterpret_cast<const float4 *>(src);
    const float4 hi = *reinterpret_cast<const float4 *>(src + D / 2);
    const int tp = pos[b];
    const bool live = flat < B * heads && tp >= 0 && tp < T_cap;
    // first token of the 64-token block that holds tp: in the sequence's own row, or in its page of the pool
    int64_t blk0 = ((int64_t)b * Hkv + h) * T_cap + (tp & ~63);
    if (block_table && live && !is_q) blk0 = ((int64_t)block_table[(int64_t)b * max_pages + (tp >> 6)] * Hkv + h) * 64;
    float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    if constexpr (ROPE) {
        if (live && !is_v) {
            const float4 c4 = *reinterpret_cast<const float4 *>(cs + (int64_t)tp * (D / 2) + 4 * j);
            const float4 s4 = *reinterpret_cast<const float4 *>(sn + (int64_t)tp * (D / 2) + 4 * j);
            rope8(v, c4, s4);
            if (is_q) {
                float *dst = q_out + ((int64_t)b * Hq + hd) * D + 4 * j;
                *reinterpret_cast<float4 *>(dst) = make_float4(v[0], v[1], v[2], v[3]);
                *reinterpret_cast<float4 *>(dst + D / 2) = make_float4(v[4], v[5], v[6], v[7]);
            }
        }
    }
    fwht_codes<D>(v, j);   // every lane takes part in the cross-lane stages
    const float a = max_lanes<LPB>(abs8(v));
    const float sc = (a == 0.0f) ? 1.0f : a / 127.0f;
    const float inv = (a == 0.0f) ? 0.0f : 127.0f / a;
    if (live && !is_q) {
        const uint32_t c0 = quant4(v[0], v[1], v[2], v[3], inv), c1 = quant4(v[4], v[5], v[6], v[7], inv);
        if (j == 0) (is_v ? vs : ks)[blk0 + (tp & 63)] = sc;
        store_token(is_v, j, tp, blk0, c0, c1, kq, vt);
    }
}

constexpr int NT_MAX = 4;

struct Plan {
    int splits, per;   // workgroups per cache row, 64-token blocks per workgroup
    int waves;         // of a workgroup: 4, or 8 where it sees a whole sequence
};

int max_splits(int64_t B, int64_t Hkv, int64_t T);

// How many spans a row is cut into, of equal length but for the last.  Where 16 blocks a workgroup (four a wave) do not give
// every compute unit a workgroup: a block for each of a workgroup's waves, or two, three or four where these workgroups are more
// than the units or, with codes, their spans more than the merge reads at once; and no cut at all up to eight blocks where the
// workgroup then writes the output itself.  (Cut until every unit had a workgroup, a span was a block or two, most waves had
// nothing to do and the merge was the longer half.  us of attention and merge before -> after, 8 heads: one sequence of 300 tokens
// 7.2 -> 5.8, of 700 10.7 -> 7.0, of 1531 9.0 -> 7.5, of 4096 9.5 -> 8.1; 2 of 500 7.8 -> 6.3, 4 of 2500 11.2 -> 9.9; with codes,
// one of 1531 14.3 -> 8.1, 4 of 1024 9.2 -> 8.0.)  Else the count whose busiest unit is done first, at four
// blocks a wave or fewer: workgroups a unit times the blocks that a workgroup streams and START more for its start and end; the
// merge counts as MERGE blocks of a unit, a quarter more for every span and BATCH for every further batch of loads that it makes,
// and a finer cut has to promise a tenth (for a twentieth, mixed lengths lose what equal ones gain: 20 sequences of up to 3907
// tokens 0.96 and 1.05 times the time).  Fitted to timings of all cuts of 92 shapes, 500 to 60000 tokens, equal and mixed lengths,
// rows and codes; with what it chooses there the kernels take 0.95 of the time of spans of 16 blocks throughout, 1.08 at worst.
// us with spans of 16 blocks -> here: 24 sequences of 3001 tokens 35.2 -> 31.3, of 750 to 3001 in pages 29.0 -> 24.7, 12 of 2500
// 21.4 -> 16.2, 25 of 600 to 2400 25.0 -> 19.7, 32 of 318 9.5 -> 7.1; 16 of 4096 are two workgroups a unit either way, 28.7.
// Without BATCH three sequences of 32768 were cut into 64 spans instead of 32: 39.4 instead of 25.0, the merge alone 15 more.
//
// A row of 5 to 16 blocks whose workgroup may write the output itself (`alone`) goes to one workgroup of eight waves: no merge and no
// second launch.  Up to 8 blocks the waves take one block instead of two, which pays until the rows fill three quarters of the units
// (0.90 to 0.98 of the time, recorded and replayed, 2 to 128 rows of 270 to 512 tokens).  From 9 blocks on it pays where the spans of
// four blocks that it stands for are more than the units: 9 to 12 blocks 0.88 to 0.92 at 88 to 128 rows and 1.01 to 1.10 below
// (2 sequences of 768, one head 6.7 -> 7.3 us; 21 of 704, 4 heads 8.1 -> 8.8), up to three quarters of the units (0.98 to 1.00
// at 160 to 188); 13 to 16 blocks 0.88 to 0.97 from 66 rows on and 1.07 to 1.12 at 64 (16 of 1024, 4 heads 8.4 -> 9.4; one more 8.5 -> 8.2).
// Sixteen waves took 2 us more than eight: what every wave does for itself, the queries above all, and the waves' meeting.
// (Not one sequence: it is cut alike with codes and without, see below.)
static Plan pick(int64_t B, int64_t Hq, int64_t Hkv, int64_t T, bool quant, bool alone)
{
    constexpr int START = 3, MERGE = 5, BATCH = 4, DIRECT = 8;
    const int blocks = (int)((T + 63) / 64);
    const int64_t rows = B * Hkv, cus = compute_units();
    Plan pl;
    pl.waves = 4;
    const int fewest = (blocks + 4 * NT_MAX - 1) / (4 * NT_MAX);
    if (alone && B > 1 && blocks > 4 && blocks <= 16 && (blocks <= 8 || rows * ((blocks + 3) / 4) > cus) &&
        (blocks <= 12 ? 4 * rows < 3 * cus : rows < cus)) {
        pl.splits = 1;
        pl.per = blocks;
        pl.waves = 8;
        return pl;
    }
    if (rows * fewest < cus) {
        // (one sequence is cut alike with codes and without: the call with the projection makes its codes either way)
        const bool codes = quant && B > 1;
        if (!codes && blocks <= DIRECT) pl.per = blocks;
        else {
            const int64_t most = codes ? 8 : cus;
            auto spans = [&] { return (int64_t)((blocks + pl.per - 1) / pl.per); };
            for (pl.per = 4; pl.per < 4 * NT_MAX && (rows * spans() > cus || spans() > most); pl.per += 4) {}
        }
        pl.splits = (blocks + pl.per - 1) / pl.per;
        return pl;
    }
    // (a span takes whole rounds of its waves: one of 13 blocks is as long as one of 16, and loads blocks of the next.  31 sequences
    // of 3199 tokens in pages 24.3 us in spans of 16, 16, 16 and 2 blocks, 26.0 in 13, 13, 13 and 11)
    auto cut4 = [&](int s) { pl.per = ((blocks + s - 1) / s + 3) / 4 * 4, pl.splits = (blocks + pl.per - 1) / pl.per; };
    auto cost = [&]() -> int64_t {   // in quarters
        const int64_t stream = (rows * pl.splits + cus - 1) / cus * (pl.per + START);
        const int merge = pl.splits > 1 ? MERGE + BATCH * (attn::merge_batches(pl.splits, B * Hq, quant) - 1) : 0;
        return 4 * (stream + merge) + (pl.splits > 1 ? pl.splits : 0);
    };
    // (no more of them than the workspace was sized for before)
    const int most = std::min(std::max(max_splits(B, Hkv, T), attn::max_splits(B, Hkv, T)), (blocks + 7) / 8);
    cut4(fewest);
    int best = fewest;
    const int64_t first = cost();
    int64_t best_cost = first;
    for (int s = fewest + 1; s <= most; ++s) {
        cut4(s);
        const int64_t c = cost();
        if (10 * c < 9 * first && c < best_cost) best = s, best_cost = c;
    }
    cut4(best);
    return pl;
}

// At least the largest split count of the plans above for any length in [1, T]: what workspaces are sized for.  For few rows it is
// the count of an earlier plan, which cut until every unit had a workgroup, up to four times what the present one uses, and stays so
// that a workspace is the size it has always been.
int max_splits(int64_t B, int64_t Hkv, int64_t T)
{
    const int blocks = (int)((T + 63) / 64);
    const int64_t rows = B * Hkv, cus = compute_units();
    int best = (blocks + 4 * NT_MAX - 1) / (4 * NT_MAX);
    int want = (int)((cus + rows - 1) / rows);
    if (want > blocks) want = blocks;
    if (rows < cus && want > best) best = want;
    return best;
}

}  // namespace avt
}  // namespace mi

using namespace mi;

static int64_t align_up(int64_t v, int64_t a) { return (v + a - 1) / a * a; }

// the decode step's rotary embedding and append, done by the attention kernel itself
struct StepIn {
    const float *qkv;
    int64_t stride;
    const float *cs, *sn;
    const int32_t *pos;
};

// the partial results of a call whose caller merges them itself, where it may (splits 0: they have been merged, or never were)
struct Unmerged {
    int64_t N;   // columns of the projection behind it
    const float *o, *ml;
    int splits;
};

struct ScoreGate {
    int8_t *qq;
    float *sq;
    int32_t *dots;
};

static int32_t run_tiled(const float *q, const int8_t *kq, const float *ks, const int8_t *vt, const float *vs, float *o,
                      int8_t *oq, float *oscale, int64_t B, int64_t Hq, int64_t Hkv, int64_t D, int64_t T_cap,
                      const int32_t *seq_len, int64_t T_max, int32_t out_rotated, void *workspace,
                      int64_t workspace_bytes, hipStream_t s, const int32_t *block_table = nullptr,
                      int64_t max_pages = 0, const ScoreGate *dbg = nullptr, const StepIn *step = nullptr,
                      Unmerged *unmerged = nullptr)
{
    if (block_table) {   // paged: the capacity of a sequence is its share of the table
        if (max_pages <= 0 || max_pages > (1 << 18) || !seq_len || !aligned4(block_table)) return MI_EINVAL;
        T_cap = max_pages * 64;
    }
    if (B <= 0 || Hq <= 0 || Hkv <= 0 || T_cap <= 0 || T_max <= 0 || T_max > T_cap) return MI_EINVAL;
    if (D != avt::D || Hq % Hkv || Hq / Hkv > 4 || T_cap % 64) return MI_EINVAL;
    if (T_cap > (1LL << 24) || B * Hkv > 65535) return MI_ERANGE;
    if (!q || !kq || !ks || !vt || !vs || !workspace) return MI_EINVAL;
    if (!aligned16(q) || !aligned16(kq) || !aligned16(vt) || !aligned16(ks) || !aligned16(vs) || !aligned16(workspace))
        return MI_EINVAL;
    if (seq_len && !aligned4(seq_len)) return MI_EINVAL;
    if (workspace_bytes < mi_gqa_decode_workspace_bytes(B, Hq, Hkv, D, T_max)) return MI_ENOSPC;
    // where one workgroup sees the whole sequence it may write the output rows (the gate takes the split form: it wants no o)
    const int64_t obytes = B * Hq * D * 4;   // (on top of the queries: row by row, or with a merge)
    const bool alone = !oq && !dbg && (o == q || !overlaps(o, obytes, q, obytes));
    const avt::Plan plan = avt::pick(B, Hq, Hkv, T_max, oq != nullptr, alone && !step);   // (a step of several sequences asks for codes)
    const bool direct = plan.splits == 1 && alone;
    avt::StepParams p = {};
    p.q = q; p.kq = kq; p.ks = ks; p.vt = vt; p.vs = vs;
    p.Hq = (int)Hq; p.Hkv = (int)Hkv; p.G = (int)(Hq / Hkv); p.T = (int)T_max;
    p.Tstride = (int)T_cap;
    p.splits = plan.splits;
    p.seq_len = seq_len;
    p.score_scale = 1.4426950408889634f * 0.08838834764831845f;  // log2(e) / sqrt(128)
    p.o = o; p.out_rotated = out_rotated;
    p.block_table = block_table; p.max_pages = (int)max_pages;
    p.dbg_qq = dbg ? dbg->qq : nullptr;
    p.dbg_sq = dbg ? dbg->sq : nullptr;
    p.dbg_dots = dbg ? dbg->dots : nullptr;
    p.part_o = static_cast<float *>(workspace);
    p.part_ml = reinterpret_cast<float *>(static_cast<char *>(workspace) +
                                          align_up(B * Hkv * plan.splits * 4 * avt::D * 4, 256));
    if (step) {
        p.qkv = step->qkv; p.qkv_stride = step->stride; p.cs = step->cs; p.sn = step->sn; p.pos = step->pos;
    }
    p.blocks_per_split = plan.per;
    const dim3 grid((unsigned)plan.splits, (unsigned)(B * Hkv));
    const int nt = (plan.per + plan.waves - 1) / plan.waves;
    // (p as its base without APPEND)
    if (plan.waves == 8) {
        if (nt <= 1) launch_kernel((avt::k_gqa_tiled_split<8, 1, 8, true, false>), grid, dim3(512), 0, s, p);
        else launch_kernel((avt::k_gqa_tiled_split<8, 2, 8, true, false>), grid, dim3(512), 0, s, p);
        return launch_status();
    }
#define MI_TILED(NT_, DIR_, APP_) launch_kernel((avt::k_gqa_tiled_split<4, NT_, 8, DIR_, APP_>), grid, dim3(256), 0, s, p)
#define MI_TILED_NT(DIR_, APP_) do { if (nt <= 1) MI_TILED(1, DIR_, APP_); else if (nt <= 2) MI_TILED(2, DIR_, APP_); else if (nt <= 3) MI_TILED(3, DIR_, APP_); else MI_TILED(4, DIR_, APP_); } while (0)
    if (step) { if (direct) MI_TILED_NT(true, true); else MI_TILED_NT(false, true); }
    else { if (direct) MI_TILED_NT(true, false); else MI_TILED_NT(false, false); }
#undef MI_TILED_NT
#undef MI_TILED
    if (direct || dbg) return launch_status();
    int32_t rc = launch_status();
    if (rc) return rc;
    if (unmerged && merged_takes(plan.splits, unmerged->N, Hq * D)) {
        unmerged->o = p.part_o;
        unmerged->ml = p.part_ml;
        unmerged->splits = plan.splits;
        return MI_OK;
    }
    return attn::launch_merge(p.part_o, p.part_ml, o, oq, oscale, B, Hq, Hkv, plan.splits, out_rotated, s);
}

extern "C" int32_t mi_gqa_decode_attn_tiled(const float *q, const int8_t *kq, const float *ks, const int8_t *vt,
                                         const float *vs, float *o, int64_t B, int64_t Hq, int64_t Hkv, int64_t D,
                                         int64_t T_cap, const int32_t *seq_len, int64_t T_max, int32_t out_rotated,
                                         void *workspace, int64_t workspace_bytes, void *stream)
{
    if (!o || !aligned16(o)) return MI_EINVAL;
    return run_tiled(q, kq, ks, vt, vs, o, nullptr, nullptr, B, Hq, Hkv, D, T_cap, seq_len, T_max, out_rotated, workspace,
                  workspace_bytes, as_stream(stream));
}

extern "C" int32_t mi_gqa_decode_attn_tiled_quant_i8(const float *q, const int8_t *kq, const float *ks, const int8_t *vt,
                                                  const float *vs, float *o_rot, int8_t *oq, float *oscale, int64_t B,
                                                  int64_t Hq, int64_t Hkv, int64_t D, int64_t T_cap,
                                                  const int32_t *seq_len, int64_t T_max, void *workspace,
                                                  int64_t workspace_bytes, void *stream)
{
    if (!oq || !oscale || !aligned4(oq) || !aligned4(oscale) || (o_rot && !aligned16(o_rot))) return MI_EINVAL;
    if (Hq > 64) return MI_ERANGE;
    return run_tiled(q, kq, ks, vt, vs, o_rot, oq, oscale, B, Hq, Hkv, D, T_cap, seq_len, T_max, 1, workspace,
                  workspace_bytes, as_stream(stream));
}

// Gate helper for this layout: the split kernel alone, which also writes out the int8 query codes, their scales and
// the raw int32 dots it works from (no merge, no o).
extern "C" int32_t mi_gqa_decode_scores_tiled_i32(const float *q, const int8_t *kt, const float *ks, const int8_t *vt,
                                                  const float *vs, int8_t *qq, float *sq, int32_t *dots, int64_t B,
                                                  int64_t Hq, int64_t Hkv, int64_t D, int64_t T_cap, int64_t T,
                                                  void *workspace, int64_t workspace_bytes, void *stream)
{
    if (!qq || !sq || !dots || !aligned4(qq) || !aligned4(sq) || !aligned4(dots)) return MI_EINVAL;
    const ScoreGate g = {qq, sq, dots};
    return run_tiled(q, kt, ks, vt, vs, nullptr, nullptr, nullptr, B, Hq, Hkv, D, T_cap, nullptr, T, 1, workspace,
                     workspace_bytes, as_stream(stream), nullptr, 0, &g);
}

namespace mi {
int32_t launch_merged_linear(const float *, const float *, int, int, const int8_t *, const float *, float *, float *, int8_t *, float *,
                             int64_t, int64_t, hipStream_t);
int32_t launch_linear_fused(const float *, const int8_t *, const float *, float *, int8_t *, float *, int64_t, int64_t,
                            int64_t, hipStream_t, bool);
}

// Attention and the output projection behind it as one call.  Workspace: the merged rows (fp32, rotated basis), their
// codes and their scales (offsets that depend on B and Hq alone), then the attention's own.
extern "C" int64_t mi_gqa_decode_attn_linear_workspace_bytes(int64_t B, int64_t Hq, int64_t Hkv, int64_t D, int64_t T)
{
    const int64_t a = mi_gqa_decode_workspace_bytes(B, Hq, Hkv, D, T);
    if (a < 0) return a;
    return a + align_up(B * Hq * D * 4, 256) + align_up(B * Hq * D, 256) + align_up(B * 4, 256);
}

static int32_t attn_linear(const float *q, const int8_t *kq, const float *ks, const int8_t *vt, const float *vs, float *o_rot,
                           const int8_t *qw, const float *sw, float *y, int64_t B, int64_t Hq, int64_t Hkv, int64_t D,
                           int64_t T_cap, const int32_t *seq_len, int64_t T_max, int64_t N, void *workspace,
                           int64_t workspace_bytes, void *stream, const StepIn *step)
{
    if (!qw || !sw || !y || !workspace || N <= 0 || N % 16) return MI_EINVAL;
    if (!aligned16(qw) || !aligned16(sw) || !aligned16(y) || !aligned16(workspace) || (o_rot && !aligned16(o_rot)))
        return MI_EINVAL;
    if (Hq > 64) return MI_ERANGE;
    const int64_t attn_bytes = mi_gqa_decode_workspace_bytes(B, Hq, Hkv, D, T_max);
    if (attn_bytes < 0) return (int32_t)attn_bytes;
    if (workspace_bytes < mi_gqa_decode_attn_linear_workspace_bytes(B, Hq, Hkv, D, T_max)) return MI_ENOSPC;
    const int64_t K = Hq * D;
    char *base = static_cast<char *>(workspace);
    float *row = reinterpret_cast<float *>(base);
    int8_t *oq = reinterpret_cast<int8_t *>(base + align_up(B * K * 4, 256));
    float *oscale = reinterpret_cast<float *>(reinterpret_cast<char *>(oq) + align_up(B * K, 256));
    void *attn_ws = reinterpret_cast<char *>(oscale) + align_up(B * 4, 256);
    hipStream_t s = as_stream(stream);
    float *orow = o_rot ? o_rot : row;
    if (B == 1 && K >= 1024 && row_takes(N, K) && apart({{orow, K * 4}}, {{y, N * 4}, {oq, K}, {oscale, 4}})) {
        // One token: merging its Hq rows AND quantizing them in one workgroup makes that workgroup read every split's
        // partials (Hq x splits x 512 B, half a megabyte at 32 splits) through one compute unit.  Here the merge runs
        // over many workgroups and leaves the fp32 row; the projection's GEMV quantizes it in its own prologue
        // (the same row quantizer on the same values: identical codes, scale and y).  Its workgroups read the row while
        // others write: an output on top of the row takes the other route.  So do rows of less than eight heads, whose merge has
        // the fewest workgroups (four heads, 4000 tokens, 4096 outputs 24.2 us there, 25.1 here; eight heads 27.1 and 26.1).
        // Up to eight splits the GEMV merges them as well, and leaves the row in the workspace (a row of the caller's may lie
        // on what the others still read).
        Unmerged parts = {N, nullptr, nullptr, 0};
        const bool may = !o_rot && apart({{attn_ws, attn_bytes}}, {{y, N * 4}});
        int32_t rc = run_tiled(q, kq, ks, vt, vs, orow, nullptr, nullptr, B, Hq, Hkv, D, T_cap, seq_len, T_max, 1, attn_ws,
                               attn_bytes, s, nullptr, 0, nullptr, step, may ? &parts : nullptr);
        if (rc) return rc;
        if (parts.splits)
            return launch_merged_linear(parts.o, parts.ml, parts.splits, (int)(Hq / Hkv), qw, sw, y, row, oq, oscale, N, K, s);
        return launch_linear_fused(orow, qw, sw, y, oq, oscale, 1, N, K, s, false);
    }
    int32_t rc = run_tiled(q, kq, ks, vt, vs, o_rot, oq, oscale, B, Hq, Hkv, D, T_cap, seq_len, T_max, 1, attn_ws,
                           attn_bytes, s, nullptr, 0, nullptr, step);
    if (rc) return rc;
    return mi_w8a8_gemm_dequant_f32(oq, oscale, qw, sw, y, B, N, K, stream);
}

extern "C" int32_t mi_gqa_decode_attn_tiled_linear_f32(const float *q, const int8_t *kq, const float *ks,
                                                       const int8_t *vt, const float *vs, float *o_rot,
                                                       const int8_t *qw, const float *sw, float *y, int64_t B,
                                                       int64_t Hq, int64_t Hkv, int64_t D, int64_t T_cap,
                                                       const int32_t *seq_len, int64_t T_max, int64_t N,
                                                       void *workspace, int64_t workspace_bytes, void *stream)
{
    return attn_linear(q, kq, ks, vt, vs, o_rot, qw, sw, y, B, Hq, Hkv, D, T_cap, seq_len, T_max, N, workspace,
                       workspace_bytes, stream, nullptr);
}

extern "C" int32_t mi_kv_tiled_from_rows_i8(const int8_t *kq, const int8_t *vq, int8_t *kt, int8_t *vt, int64_t rows,
                                            int64_t T, int64_t src_stride, int64_t T_cap, void *stream)
{
    if ((!kq && !vq) || (kq && !kt) || (vq && !vt)) return MI_EINVAL;
    if (rows <= 0 || T <= 0 || T > src_stride || T > T_cap || T_cap % 64) return MI_EINVAL;
    if ((kq && (!aligned16(kq) || !aligned16(kt))) || (vq && (!aligned16(vq) || !aligned16(vt)))) return MI_EINVAL;
    if (rows > 65535 || T_cap > (1LL << 24)) return MI_ERANGE;
    const unsigned blocks = (unsigned)((T + 63) / 64);
    const dim3 grid(blocks, (unsigned)rows, (kq && vq) ? 2 : 1);
    launch_kernel(avt::k_tiled_from_rows, grid, dim3(256), 0, as_stream(stream), kq, vq, kt, vt, (int)T, src_stride,
                  T_cap, (kq ? 0 : 1));
    return launch_status();
}

static int32_t check_append(const void *a, const void *b, const void *kq, const void *ks, const void *vt,
                            const void *vs, const void *pos, int64_t B, int64_t Hkv, int64_t D, int64_t T_cap)
{
    if (!a || !b || !kq || !ks || !vt || !vs || !pos) return MI_EINVAL;
    if (B <= 0 || Hkv <= 0 || T_cap <= 0 || T_cap % 64 || D != 128) return MI_EINVAL;
    if (B * Hkv > (1LL << 24) || T_cap > (1LL << 24)) return MI_ERANGE;
    if (!aligned16(a) || !aligned16(b) || !aligned4(kq) || !aligned4(ks) || !aligned4(vs) || !aligned4(pos))
        return MI_EINVAL;
    return MI_OK;
}

extern "C" int32_t mi_kv_append_tiled_f32_i8(const float *k_new, const float *v_new, int64_t row_stride, int8_t *kq,
                                          float *ks, int8_t *vt, float *vs, const int32_t *pos, int64_t B,
                                          int64_t Hkv, int64_t D, int64_t T_cap, void *stream)
{
    int32_t rc = check_append(k_new, v_new, kq, ks, vt, vs, pos, B, Hkv, D, T_cap);
    if (rc) return rc;
    if (row_stride < Hkv * D || row_stride % 4) return MI_EINVAL;
    const dim3 grid((unsigned)((B * Hkv + 15) / 16), 2);
    launch_kernel(avt::k_kv_append_vt<false>, grid, dim3(256), 0, as_stream(stream), k_new, v_new, row_stride,
                  (const float *)nullptr, (const float *)nullptr, (float *)nullptr, kq, ks, vt, vs, pos, (int)B, 0,
                  (int)Hkv, (int)T_cap, (const int32_t *)nullptr, 0);
    return launch_status();
}

extern "C" int32_t mi_rope_kv_append_tiled_f32_i8(const float *qkv, int64_t row_stride, const float *rope_cos,
                                               const float *rope_sin, float *q_out, int8_t *kq, float *ks,
                                               int8_t *vt, float *vs, const int32_t *pos, int64_t B, int64_t Hq,
                                               int64_t Hkv, int64_t D, int64_t T_cap, void *stream)
{
    int32_t rc = check_append(qkv, q_out, kq, ks, vt, vs, pos, B, Hkv, D, T_cap);
    if (rc) return rc;
    if (!rope_cos || !rope_sin || !aligned16(rope_cos) || !aligned16(rope_sin) || Hq <= 0) return MI_EINVAL;
    if (row_stride < (Hq + 2 * Hkv) * D || row_stride % 4) return MI_EINVAL;
    const int64_t heads = B * (Hq + 2 * Hkv);
    launch_kernel(avt::k_kv_append_vt<true>, dim3((unsigned)((heads + 15) / 16)), dim3(256), 0, as_stream(stream),
                  qkv, (const float *)nullptr, row_stride, rope_cos, rope_sin, q_out, kq, ks, vt, vs, pos, (int)B,
                  (int)Hq, (int)Hkv, (int)T_cap, (const int32_t *)nullptr, 0);
    return launch_status();
}

extern "C" int32_t mi_rope_append_attn_tiled_linear_f32(const float *qkv, int64_t row_stride, const float *rope_cos,
                                                        const float *rope_sin, float *q_out, int8_t *kq, float *ks,
                                                        int8_t *vt, float *vs, const int32_t *pos, float *o_rot,
                                                        const int8_t *qw, const float *sw, float *y, int64_t B,
                                                        int64_t Hq, int64_t Hkv, int64_t D, int64_t T_cap,
                                                        const int32_t *seq_len, int64_t T_max, int64_t N,
                                                        void *workspace, int64_t workspace_bytes, void *stream)
{
    int32_t rc = check_append(qkv, q_out, kq, ks, vt, vs, pos, B, Hkv, D, T_cap);
    if (rc) return rc;
    if (!rope_cos || !rope_sin || !aligned16(rope_cos) || !aligned16(rope_sin) || Hq <= 0) return MI_EINVAL;
    if (row_stride < (Hq + 2 * Hkv) * D || row_stride % 4) return MI_EINVAL;
    // The attention kernel stores rows of q_out (and, with one split, of o_rot) while other workgroups still read qkv, and
    // both in no order among each other: a caller whose buffers overlap gets the two launches.
    const int64_t out_bytes = B * Hq * D * 4, qkv_bytes = ((B - 1) * row_stride + (Hq + 2 * Hkv) * D) * 4;
    if (overlaps(q_out, out_bytes, qkv, qkv_bytes) || overlaps(o_rot, out_bytes, qkv, qkv_bytes) ||
        overlaps(o_rot, out_bytes, q_out, out_bytes)) {
        rc = mi_rope_kv_append_tiled_f32_i8(qkv, row_stride, rope_cos, rope_sin, q_out, kq, ks, vt, vs, pos, B, Hq, Hkv, D,
                                            T_cap, stream);
        if (rc) return rc;
        return attn_linear(q_out, kq, ks, vt, vs, o_rot, qw, sw, y, B, Hq, Hkv, D, T_cap, seq_len, T_max, N, workspace,
                           workspace_bytes, stream, nullptr);
    }
    const StepIn step = {qkv, row_stride, rope_cos, rope_sin, pos};
    return attn_linear(q_out, kq, ks, vt, vs, o_rot, qw, sw, y, B, Hq, Hkv, D, T_cap, seq_len, T_max, N, workspace,
                       workspace_bytes, stream, &step);
}

// ---- the paged form of the tiled cache: pools of 64-token pages, one page = one 8 KB key block (four 16-token tiles)
// and one 8 KB transposed value block per kv head, so the attention kernel's loads stay 1 KB contiguous and a block
// costs it one scalar table look-up.
extern "C" int32_t mi_gqa_decode_attn_tiled_paged(const float *q, const int8_t *kt_pool, const float *ks_pool,
                                                  const int8_t *vt_pool, const float *vs_pool, float *o,
                                                  const int32_t *block_table, int64_t max_pages, int64_t B,
                                                  int64_t Hq, int64_t Hkv, int64_t D, const int32_t *seq_len,
                                                  int64_t T_max, int32_t out_rotated, void *workspace,
                                                  int64_t workspace_bytes, void *stream)
{
    if (!o || !aligned16(o) || !block_table) return MI_EINVAL;
    return run_tiled(q, kt_pool, ks_pool, vt_pool, vs_pool, o, nullptr, nullptr, B, Hq, Hkv, D, 0, seq_len, T_max,
                     out_rotated, workspace, workspace_bytes, as_stream(stream), block_table, max_pages);
}

extern "C" int32_t mi_gqa_decode_attn_tiled_paged_quant_i8(const float *q, const int8_t *kt_pool, const float *ks_pool,
                                                           const int8_t *vt_pool, const float *vs_pool, float *o_rot,
                                                           int8_t *oq, float *oscale, const int32_t *block_table,
                                                           int64_t max_pages, int64_t B, int64_t Hq, int64_t Hkv,
                                                           int64_t D, const int32_t *seq_len, int64_t T_max,
                                                           void *workspace, int64_t workspace_bytes, void *stream)
{
    if (!oq || !oscale || !aligned4(oq) || !aligned4(oscale) || (o_rot && !aligned16(o_rot)) || !block_table) return MI_EINVAL;
    if (Hq > 64) return MI_ERANGE;
    return run_tiled(q, kt_pool, ks_pool, vt_pool, vs_pool, o_rot, oq, oscale, B, Hq, Hkv, D, 0, seq_len, T_max, 1,
                     workspace, workspace_bytes, as_stream(stream), block_table, max_pages);
}

extern "C" int32_t mi_kv_append_tiled_paged_f32_i8(const float *k_new, const float *v_new, int64_t row_stride,
                                                   int8_t *kt_pool, float *ks_pool, int8_t *vt_pool, float *vs_pool,
                                                   const int32_t *block_table, int64_t max_pages, const int32_t *pos,
                                                   int64_t B, int64_t Hkv, int64_t D, void *stream)
{
    if (!block_table || !aligned4(block_table) || max_pages <= 0 || max_pages > (1 << 18)) return MI_EINVAL;
    int32_t rc = check_append(k_new, v_new, kt_pool, ks_pool, vt_pool, vs_pool, pos, B, Hkv, D, max_pages * 64);
    if (rc) return rc;
    if (row_stride < Hkv * D || row_stride % 4) return MI_EINVAL;
    const dim3 grid((unsigned)((B * Hkv + 15) / 16), 2);
    launch_kernel(avt::k_kv_append_vt<false>, grid, dim3(256), 0, as_stream(stream), k_new, v_new, row_stride,
                  (const float *)nullptr, (const float *)nullptr, (float *)nullptr, kt_pool, ks_pool, vt_pool,
                  vs_pool, pos, (int)B, 0, (int)Hkv, (int)(max_pages * 64), block_table, (int)max_pages);
    return launch_status();
}

extern "C" int32_t mi_rope_kv_append_tiled_paged_f32_i8(const float *qkv, int64_t row_stride, const float *rope_cos,
                                                        const float *rope_sin, float *q_out, int8_t *kt_pool,
                                                        float *ks_pool, int8_t *vt_pool, float *vs_pool,
                                                        const int32_t *block_table, int64_t max_pages,
                                                        const int32_t *pos, int64_t B, int64_t Hq, int64_t Hkv,
                                                        int64_t D, void *stream)
{
    if (!block_table || !aligned4(block_table) || max_pages <= 0 || max_pages > (1 << 18)) return MI_EINVAL;
    int32_t rc = check_append(qkv, q_out, kt_pool, ks_pool, vt_pool, vs_pool, pos, B, Hkv, D, max_pages * 64);
    if (rc) return rc;
    if (!rope_cos || !rope_sin || !aligned16(rope_cos) || !aligned16(rope_sin) || Hq <= 0) return MI_EINVAL;
    if (row_stride < (Hq + 2 * Hkv) * D || row_stride % 4) return MI_EINVAL;
    const int64_t heads = B * (Hq + 2 * Hkv);
    launch_kernel(avt::k_kv_append_vt<true>, dim3((unsigned)((heads + 15) / 16)), dim3(256), 0, as_stream(stream),
                  qkv, (const float *)nullptr, row_stride, rope_cos, rope_sin, q_out, kt_pool, ks_pool, vt_pool,
                  vs_pool, pos, (int)B, (int)Hq, (int)Hkv, (int)(max_pages * 64), block_table, (int)max_pages);
    return launch_status();
}
