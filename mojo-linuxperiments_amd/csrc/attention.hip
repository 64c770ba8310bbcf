// Grouped-query decode attention over an int8 KV cache (workload element a8).
//
//   per (b, h):  q' = quant(FWHT128(q))            int8 codes qq, scale sq
//                dot_t = qq . kq[b, h/G, t, :]      int32
//                s_t = dot_t * sq * ks_t / sqrt(D)
//                o' = sum_t softmax(s)_t * vs_t * vq[b, h/G, t, :]
//   and, unless the caller wants the rotated basis, o = FWHT128(o').
//
// Split-KV: grid = (splits, B*Hkv); a workgroup (4 waves) streams one span of
// tokens of one KV head once and serves the G = Hq/Hkv <= 4 query heads that
// share it.  A second small kernel merges the splits.
//
// Pass 1 (scores).  Keys are loaded straight in MFMA operand layout (lane l: token l%16 of a 16-token tile,
// 16-byte chunk l/16 of each half of the head dimension); two v_mfma_i32_16x16x64_i8 per tile against the
// query codes of the G heads give the exact int32 dot products (lane l < 16: token l, register r: head r).
// Scores (already in log2 units) go to LDS, the running max stays in registers.
// Pass 2 (P.V).  v_mfma_f32_4x4x1_16B_f32 treats each aligned group of
// four lanes as one 4x4 outer product: the four lanes share a token, lane
// l%4 = i supplies p(token, head i) * vs(token) as the A value and one V
// element as the B value, so register i of the accumulator is head i.  Sixteen
// such MFMAs (one per byte of the lane's 16) consume a load; int8 -> fp32 is
// one v_cvt_f32_i32 that selects its byte.  The fp32 matrix pipe does the 4-head FMA work that would
// otherwise cost 64 VALU FMAs per 16 bytes.
//
// Bound: HBM.  Algorithmic bytes = K and V codes (2*B*Hkv*T*D) + their scales
// (8*B*Hkv*T) + q and o (8*B*Hq*D).
#include "attn_merge.h"
#include "fwht_core.h"

namespace mi {

namespace avt {
int max_splits(int64_t B, int64_t Hkv, int64_t T);   // attention_tiled.hip: the block-transposed V layout's own plan
}

namespace attn {

constexpr int D = 128;

__device__ __forceinline__ void fwht128(float (&v)[8], int j) { fwht_chunk<D>(v, j); }   // fwht_core.h

struct Params {
    const float *q;
    const int8_t *kq;
    const float *ks;
    const int8_t *vq;
    const float *vs;
    float *part_o;   // [B*Hkv, splits, 4, 128]
    float *part_ml;  // [B*Hkv, splits, 2, 4]   (max in log2 units, sum)
    int8_t *dump_qq;
    float *dump_sq;
    int32_t *dump_dots;
    int Hq, Hkv, G, T;    // T: tokens per sequence (the longest one when seq_len is given)
    int Tstride;          // tokens between consecutive (batch, kv head) rows of the cache
    const int32_t *seq_len;   // per-sequence token counts [B] (device), or null: every sequence holds T tokens
    const int32_t *block_table;   // paged cache: page of tokens [i*P, (i+1)*P) of sequence b at [b*max_pages + i], or null
    int max_pages, page_shift;    // P = 1 << page_shift tokens per page, P >= 16
    int tiles_per_split;  // 16-token tiles
    float score_scale;    // log2(e) / sqrt(D)
    int out_rotated;      // DIRECT kernels: leave the rows in the rotated basis of V; they are the output [B, Hq, 128], at part_o
};

// one round of the transposed butterfly over token slots: keep the half of the values whose index bit
// matches this lane's OFF bit, hand the other half to lane ^ OFF
template <int V, int OFF>
__device__ __forceinline__ void fold_slots(float (&p)[64], int lane)
{
    const bool hi = (lane & OFF) != 0;
#pragma unroll
    for (int i = 0; i < V / 2; ++i) {
        if constexpr (OFF == 32) {   // the exchange is one instruction
            const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(p[i]), __float_as_uint(p[i + V / 2]), false, false);
            p[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
        } else if constexpr (OFF == 16) {
            const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(p[i]), __float_as_uint(p[i + V / 2]), false, false);
            p[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
        } else {
            const float keep = hi ? p[i + V / 2] : p[i];
            const float send = hi ? p[i] : p[i + V / 2];
            p[i] = keep + __int_as_float(xor_lane_i<OFF>(__float_as_int(send)));
        }
    }
}

// 16-token tiles per wave: a workgroup covers at most 4 * tiles * 16 tokens.  Every wave runs through all of its
// tiles (the ones past the end masked), so a workgroup wants a span it can fill: 11 tiles (704 tokens) when there
// are (batch, kv head) rows enough to occupy the chip with such spans, 4 tiles (256 tokens) when there are few rows
// and the cache has to be cut finer to give every compute unit work.
constexpr int TILES_LONG = 11, TILES_SHORT = 4, TILES_WIDE = 8;   // (WIDE: of eight waves)
constexpr int RING = 8;           // loads a wave keeps in flight (1 KB each); tiles per wave >= RING / 2

// RAGGED: the span a workgroup can cover runs past the end of the cache and token indices are clamped for the
// loads; otherwise every address is base + constant.  Tokens past the end of the split are masked in the scores.
// PAGED: the cache is a pool of pages [page][kv head][P tokens][128]; a 16-token tile lies in one page, so a wave
// looks up one page per tile (uniform over the wave) and lanes are clamped inside their tile.
// DIRECT: the workgroup sees the whole sequence and writes the output rows itself.  NW: its waves, four, or eight where it is DIRECT.
template <bool DUMP, bool RAGGED, bool PAGED, int WAVE_TILES, bool DIRECT, int NW>
__device__ __forceinline__ void gqa_split_body(const Params &p, const int T, int8_t (&s_q)[NW][4][D], float (&s_sq)[NW][4],
                                               float (&s_red)[NW][4][D], float (&s_sc)[NW][WAVE_TILES][16][4],
                                               float (&s_m)[NW][4], float (&s_l)[NW][4])
{
    constexpr int APART = NW * 16;   // tokens from a wave's tile to its next
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int split = blockIdx.x, bkv = blockIdx.y;
    const int b = bkv / p.Hkv, kvh = bkv % p.Hkv;
    const int G = p.G;
    const int ntiles = (T + 15) >> 4;
    const int tile_lo = split * p.tiles_per_split;
    const int tile_hi = min(tile_lo + p.tiles_per_split, ntiles);
    const int t_lo = tile_lo << 4;
    const int t_end = min(tile_hi << 4, T);   // first token this workgroup does not own
    // pass 1 lane layout (MFMA operand B): token l%16 of a 16-token tile, 16-byte chunk l/16 (+4 for the
    // second half of the head dimension); pass 2 lane layout: token slot l/8 of an 8-token group, chunk l%8
    const int tk16 = lane & 15, ck = lane >> 4;
    const int hh = lane & 3, slot = lane >> 3, chunk = lane & 7;
    const int t_wave = t_lo + wave * 16;      // first token of this wave's tile 0; tile j starts j * APART tokens further
    const int8_t *kwave = p.kq + ((int64_t)bkv * p.Tstride + t_wave) * D;
    const int8_t *vwave = p.vq + ((int64_t)bkv * p.Tstride + t_wave) * D;
    const float *kswave = p.ks + (int64_t)bkv * p.Tstride + t_wave;
    const float *vswave = p.vs + (int64_t)bkv * p.Tstride + t_wave;
    const unsigned koff = (unsigned)(tk16 * D + 16 * ck);
    // paged: row index (in tokens) of the first token of each of the wave's tiles inside the pool, and the last
    // valid token offset inside that tile (tiles past the end of the sequence fall back on its last tile and are
    // masked in the scores like any token past the end)
    int64_t trow[PAGED ? WAVE_TILES : 1];
    int tlast[PAGED ? WAVE_TILES : 1];
    if constexpr (PAGED) {
        const int last_tile = (T - 1) & ~15;
#pragma unroll
        for (int j = 0; j < WAVE_TILES; ++j) {
            const int tt = min(t_wave + j * APART, last_tile);
            const int page = __builtin_amdgcn_readfirstlane(p.block_table[(int64_t)b * p.max_pages + (tt >> p.page_shift)]);
            trow[j] = (((int64_t)page * p.Hkv + kvh) << p.page_shift) + (tt & ((1 << p.page_shift) - 1));
            tlast[j] = min(T - 1 - tt, 15);
        }
    }

    // the query row goes first: loads return in order, and the rotation of q can then run under the key loads
    const int hr = lane >> 4, jj = lane & 15;
    const int head = kvh * G + min(hr, G - 1);
    const float *qr = p.q + ((int64_t)b * p.Hq + head) * D;
    const float4 qlo = *reinterpret_cast<const float4 *>(qr + 4 * jj);
    const float4 qhi = *reinterpret_cast<const float4 *>(qr + 64 + 4 * jj);

    // ---- the wave streams its 8 key tiles (two 1 KB loads each) and then its 16 value groups (one 1 KB load
    // each) through a ring of RING register slots.  A slot is refilled as soon as it has been consumed, so RING
    // KB stay in flight per wave from the first instruction to the last and the arithmetic runs under the stream.
    v4i ring[RING];
    float ksr[RING / 2], vsr[RING];
    auto load_k = [&](int j) {   // tile j -> slots (2j) % RING, (2j+1) % RING
        if constexpr (PAGED) {
            const int64_t row = trow[j] + min(tk16, tlast[j]);
            ring[(2 * j) % RING] = *reinterpret_cast<const v4i *>(p.kq + row * D + 16 * ck);
            ring[(2 * j + 1) % RING] = *reinterpret_cast<const v4i *>(p.kq + row * D + 64 + 16 * ck);
            ksr[j % (RING / 2)] = p.ks[row];
        } else if constexpr (RAGGED) {
            const int tk = min(t_wave + j * APART + tk16, T - 1) - t_wave;
            ring[(2 * j) % RING] = *reinterpret_cast<const v4i *>(kwave + (int64_t)tk * D + 16 * ck);
            ring[(2 * j + 1) % RING] = *reinterpret_cast<const v4i *>(kwave + (int64_t)tk * D + 64 + 16 * ck);
            ksr[j % (RING / 2)] = kswave[tk];
        } else {
            ring[(2 * j) % RING] = *reinterpret_cast<const v4i *>(kwave + (koff + (unsigned)(j * APART * D)));
            ring[(2 * j + 1) % RING] = *reinterpret_cast<const v4i *>(kwave + (koff + (unsigned)(j * APART * D + 64)));
            ksr[j % (RING / 2)] = kswave[(unsigned)(j * APART) + (unsigned)tk16];
        }
    };
    auto load_v = [&](int u) {   // group u = 2*tile + half -> slot (2*WAVE_TILES + u) % RING
        const int j = u >> 1, g = u & 1;
        if constexpr (PAGED) {
            const int64_t row = trow[j] + min(g * 8 + slot, tlast[j]);
            ring[(2 * WAVE_TILES + u) % RING] = *reinterpret_cast<const v4i *>(p.vq + row * D + 16 * chunk);
            vsr[u % RING] = p.vs[row];
        } else if constexpr (RAGGED) {
            const int tk = min(t_wave + j * APART + g * 8 + slot, T - 1) - t_wave;
            ring[(2 * WAVE_TILES + u) % RING] = *reinterpret_cast<const v4i *>(vwave + (int64_t)tk * D + 16 * chunk);
            vsr[u % RING] = vswave[tk];
        } else {
            ring[(2 * WAVE_TILES + u) % RING] =
                *reinterpret_cast<const v4i *>(vwave + ((unsigned)(lane * 16) + (unsigned)(j * APART * D + g * 8 * D)));
            vsr[u % RING] = vswave[(unsigned)(j * APART + g * 8) + (unsigned)slot];
        }
    };
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < RING / 2; ++j) load_k(j);
    __builtin_amdgcn_sched_barrier(0);

    // ---- query heads of this group: every wave rotates and quantizes them for itself (no workgroup barrier)
    {
        float v[8] = {qlo.x, qlo.y, qlo.z, qlo.w, qhi.x, qhi.y, qhi.z, qhi.w};
        fwht_codes<D>(v, jj);
        const float a = max_lanes<16>(abs8(v));
        const float sc = (a == 0.0f) ? 1.0f : a / 127.0f;
        const float inv = (a == 0.0f) ? 0.0f : 127.0f / a;
        const uint32_t c0 = quant4(v[0], v[1], v[2], v[3], inv), c1 = quant4(v[4], v[5], v[6], v[7], inv);
        *reinterpret_cast<uint32_t *>(&s_q[wave][hr][4 * jj]) = c0;
        *reinterpret_cast<uint32_t *>(&s_q[wave][hr][64 + 4 * jj]) = c1;
        if (jj == 0) s_sq[wave][hr] = sc;
        if constexpr (DUMP) {
            if (split == 0 && wave == 0 && hr < G) {
                int8_t *dq = p.dump_qq + ((int64_t)b * p.Hq + head) * D;
                *reinterpret_cast<uint32_t *>(dq + 4 * jj) = c0;
                *reinterpret_cast<uint32_t *>(dq + 64 + 4 * jj) = c1;
                if (jj == 0) p.dump_sq[(int64_t)b * p.Hq + head] = sc;
            }
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // MFMA operand A: row l%16 = query head (rows >= G are zero), 16-byte chunk l/16 (+4)
    v4i qa0 = {0, 0, 0, 0}, qa1 = {0, 0, 0, 0};
    if (tk16 < G) {
        qa0 = *reinterpret_cast<const v4i *>(&s_q[wave][tk16][16 * ck]);
        qa1 = *reinterpret_cast<const v4i *>(&s_q[wave][tk16][64 + 16 * ck]);
    }
    float cq[4];     // per-head factor of the score, log2 units
#pragma unroll
    for (int h = 0; h < 4; ++h) cq[h] = h < G ? s_sq[wave][h] * p.score_scale : 0.0f;

    // ---- pass 1: scores.  Two v_mfma_i32_16x16x64_i8 per tile give the exact int32 dot products of the 16
    // tokens with the G heads; lane l < 16 holds token l, register r = head r.  Scores (log2 units) go to LDS.
    float m4[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
    for (int j = 0; j < WAVE_TILES; ++j) {
        v4i dots = __builtin_amdgcn_mfma_i32_16x16x64_i8(qa0, ring[(2 * j) % RING], (v4i){0, 0, 0, 0}, 0, 0, 0);
        dots = __builtin_amdgcn_mfma_i32_16x16x64_i8(qa1, ring[(2 * j + 1) % RING], dots, 0, 0, 0);
        const float kscale = ksr[j % (RING / 2)];
        // the two slots are free: next key tile, or the first value groups once the keys are all requested
        if (j + RING / 2 < WAVE_TILES) load_k(j + RING / 2);
        else { load_v(2 * (j + RING / 2 - WAVE_TILES)); load_v(2 * (j + RING / 2 - WAVE_TILES) + 1); }
        __builtin_amdgcn_sched_barrier(0);
        const int tt = t_wave + j * APART + tk16;
        const bool live = tt < t_end;
        float4 sc;
        sc.x = live ? (float)dots[0] * (kscale * cq[0]) : -INFINITY;
        sc.y = live ? (float)dots[1] * (kscale * cq[1]) : -INFINITY;
        sc.z = live ? (float)dots[2] * (kscale * cq[2]) : -INFINITY;
        sc.w = live ? (float)dots[3] * (kscale * cq[3]) : -INFINITY;
        if (lane < 16) {
            *reinterpret_cast<float4 *>(&s_sc[wave][j][tk16][0]) = sc;
            m4[0] = fmaxf(m4[0], sc.x); m4[1] = fmaxf(m4[1], sc.y);
            m4[2] = fmaxf(m4[2], sc.z); m4[3] = fmaxf(m4[3], sc.w);
            if constexpr (DUMP) {
                if (live) {
#pragma unroll
                    for (int h = 0; h < 4; ++h)
                        if (h < G) p.dump_dots[((int64_t)b * p.Hq + kvh * G + h) * T + tt] = dots[h];
                }
            }
        }
    }
    // maximum per head over the wave's tokens (lanes 0..15 hold partial maxima, the rest hold -inf); the softmax
    // of this wave is taken against the wave's own maximum and rescaled when the waves meet
#pragma unroll
    for (int h = 0; h < 4; ++h) {
        m4[h] = fmaxf(m4[h], __int_as_float(xor_lane_i<1>(__float_as_int(m4[h]))));
        m4[h] = fmaxf(m4[h], __int_as_float(xor_lane_i<2>(__float_as_int(m4[h]))));
        m4[h] = fmaxf(m4[h], __int_as_float(xor_lane_i<4>(__float_as_int(m4[h]))));
        m4[h] = fmaxf(m4[h], __int_as_float(xor_lane_i<8>(__float_as_int(m4[h]))));
    }
    if (lane == 0) { s_m[wave][0] = m4[0]; s_m[wave][1] = m4[1]; s_m[wave][2] = m4[2]; s_m[wave][3] = m4[3]; }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const float m_h = s_m[wave][hh];

    // ---- pass 2: P.V on the fp32 matrix pipe
    const bool counts = (lane & 4) == 0;  // each (token, head) is held by two lanes; one of them counts
    v4f acc[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = (v4f){0.f, 0.f, 0.f, 0.f};
    float lsum = 0.0f;
#pragma unroll
    for (int u = 0; u < 2 * WAVE_TILES; ++u) {
        const v4i vv = ring[(2 * WAVE_TILES + u) % RING];
        const float vscale = vsr[u % RING];
        // one conversion a code, which picks its byte and extends its sign.  (As biased bytes, v_cvt_f32_ubyte, with 128 times the
        // weights taken off at the end, the sums lost two bits: error against 64-bit
        // sums, 300 to 4096 tokens, 4.9e-7 to 8.5e-7 with it, 1.3e-7 to 1.9e-7 without; 16 sequences of 4096 tokens 29.8 and 29.2 us.)
        float f[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) f[e] = (float)(int8_t)((uint32_t)vv[e >> 2] >> (8 * (e & 3)));
        if (u + RING < 2 * WAVE_TILES) load_v(u + RING);
        __builtin_amdgcn_sched_barrier(0);
        const float score = s_sc[wave][u >> 1][8 * (u & 1) + slot][hh];
        // a wave whose tokens are all masked has m_h = -inf: exp2(-inf - -inf) would be NaN
        const float pe = (score == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(score - m_h);
        const float a = pe * vscale;
        if (counts) lsum += pe;
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[e] = __builtin_amdgcn_mfma_f32_4x4x1f32(a, f[e], acc[e], 0, 0, 0);
    }

    // sum the 8 token slots (lanes that share l%8): transposed butterfly over lane bits 5, 4, 3, after which
    // lane l holds the 8 totals with flat index 8*(l/8) .. +7, flat = 4*e + head  (56 shuffles, not 192)
    float flat[64];
#pragma unroll
    for (int e = 0; e < 16; ++e)
#pragma unroll
        for (int i = 0; i < 4; ++i) flat[4 * e + i] = acc[e][i];
    fold_slots<64, 32>(flat, lane);
    fold_slots<32, 16>(flat, lane);
    fold_slots<16, 8>(flat, lane);
    lsum = add_lane<32>(add_lane<16>(add_lane<8>(lsum)));
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int fl = 8 * slot + j;   // = 4*e + head
        s_red[wave][fl & 3][16 * chunk + (fl >> 2)] = flat[j];
    }
    if (lane < 4) s_l[wave][lane] = lsum;
    __syncthreads();

    // the waves meet: rescale each wave's sums from its own maximum to the common one
    const int64_t pbase = ((int64_t)bkv * gridDim.x + split);
    auto common = [&](int h) {
        float m = s_m[0][h];
#pragma unroll
        for (int w = 1; w < NW; ++w) m = fmaxf(m, s_m[w][h]);
        return m;
    };
    auto rescale = [&](int w, int h, float m) { return (s_m[w][h] == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(s_m[w][h] - m); };
    auto weights = [&](int h, float m) {
        float l = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; ++w) l += (s_m[w][h] == -INFINITY) ? 0.0f : s_l[w][h] * __builtin_amdgcn_exp2f(s_m[w][h] - m);
        return l;
    };
    constexpr int ADD = 64 * NW, EACH = 4 * D / ADD;   // outputs of a thread
    float total[EACH];
#pragma unroll
    for (int i = 0; i < EACH; ++i) {
        const int o = tid + ADD * i, h = o >> 7, d = o & (D - 1);
        const float m = common(h);
        if constexpr (NW == 8) {   // in pairs, and divided: 0.98 of the error of four waves and a merge against 64-bit sums (9 shapes)
            float a[8], c[8];
#pragma unroll
            for (int w = 0; w < 8; ++w) {
                const float f = rescale(w, h, m);
                a[w] = s_red[w][h][d] * f;
                c[w] = s_l[w][h] * f;
            }
            const float sum = ((a[0] + a[1]) + (a[2] + a[3])) + ((a[4] + a[5]) + (a[6] + a[7]));
            const float l = ((c[0] + c[1]) + (c[2] + c[3])) + ((c[4] + c[5]) + (c[6] + c[7]));
            total[i] = l > 0.0f ? sum / l : 0.0f;
            continue;
        }
        float sum = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; ++w) sum += s_red[w][h][d] * rescale(w, h, m);
        if constexpr (DIRECT) {
            const float l = weights(h, m);
            total[i] = l > 0.0f ? sum * (1.0f / l) : 0.0f;
        } else {
            p.part_o[(pbase * 4 + h) * D + d] = sum;
        }
    }
    if constexpr (DIRECT) {
        __syncthreads();   // every sum has been read
#pragma unroll
        for (int i = 0; i < EACH; ++i) s_red[0][(tid + ADD * i) >> 7][tid & (D - 1)] = total[i];
        __syncthreads();
        if (tid < 64 && hr < G) {   // 16 lanes per head row, as the merge kernel has them
            float *const orow = p.part_o + ((int64_t)b * p.Hq + kvh * G + hr) * D;
            float v[8];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = s_red[0][hr][4 * jj + e];
                v[4 + e] = s_red[0][hr][64 + 4 * jj + e];
            }
            if (!p.out_rotated) fwht128(v, jj);
            *reinterpret_cast<float4 *>(orow + 4 * jj) = make_float4(v[0], v[1], v[2], v[3]);
            *reinterpret_cast<float4 *>(orow + 64 + 4 * jj) = make_float4(v[4], v[5], v[6], v[7]);
        }
    } else if (tid < 4) {
        const float m = common(tid);
        p.part_ml[pbase * 8 + tid] = m;
        p.part_ml[pbase * 8 + 4 + tid] = weights(tid, m);
    }
}

template <bool DUMP, int WAVE_TILES, bool DIRECT, int NW = 4>
__global__ __launch_bounds__(64 * NW) void k_gqa_split(Params p)
{
    static_assert(NW == 4 || (NW == 8 && DIRECT), "");
    __shared__ __attribute__((aligned(16))) int8_t s_q[NW][4][D];
    __shared__ float s_sq[NW][4];
    __shared__ float s_red[NW][4][D];
    __shared__ __attribute__((aligned(16))) float s_sc[NW][WAVE_TILES][16][4];
    __shared__ float s_m[NW][4], s_l[NW][4];
    const int tile_lo = blockIdx.x * p.tiles_per_split;
    int T = p.T;
    if (p.seq_len) {
        // a cache that is filled to a different length per sequence: lengths outside [0, T] are clamped
        const int b = blockIdx.y / p.Hkv;
        T = min(max(__builtin_amdgcn_readfirstlane(p.seq_len[b]), 0), p.T);
        if (tile_lo * 16 >= T) {
            if constexpr (DIRECT) {   // a sequence of length 0: rows of zeros
                const int64_t row0 = (int64_t)b * p.Hq + (blockIdx.y % p.Hkv) * p.G;
                for (int o = threadIdx.x; o < p.G * D; o += 64 * NW) p.part_o[row0 * D + o] = 0.0f;
                return;
            }
            // this split lies past the end of the sequence: an empty partial (weight 0 in the merge)
            const int64_t pbase = ((int64_t)blockIdx.y * gridDim.x + blockIdx.x);
            for (int o = threadIdx.x; o < 4 * D; o += 256) p.part_o[pbase * 4 * D + o] = 0.0f;
            if (threadIdx.x < 4) {
                p.part_ml[pbase * 8 + threadIdx.x] = -INFINITY;
                p.part_ml[pbase * 8 + 4 + threadIdx.x] = 0.0f;
            }
            return;
        }
    }
    if (p.block_table) {
        gqa_split_body<false, true, true, WAVE_TILES, DIRECT, NW>(p, T, s_q, s_sq, s_red, s_sc, s_m, s_l);
        return;
    }
    const bool full = (tile_lo + NW * WAVE_TILES) * 16 <= T;
    if (full) gqa_split_body<DUMP, false, false, WAVE_TILES, DIRECT, NW>(p, T, s_q, s_sq, s_red, s_sc, s_m, s_l);
    else gqa_split_body<DUMP, true, false, WAVE_TILES, DIRECT, NW>(p, T, s_q, s_sq, s_red, s_sc, s_m, s_l);
}

// merge the splits of blockDim.x / 16 (b, h) rows per workgroup; 16 lanes per row.  Few rows with many splits (one
// token) take one row per workgroup, so that no compute unit reads more than one row's partials.
template <int SP>
__global__ __launch_bounds__(256) void k_gqa_merge(const float *__restrict__ part_o,
                                                   const float *__restrict__ part_ml, float *__restrict__ o,
                                                   int rows, int Hq, int Hkv, int G, int splits_rt, int out_rotated)
{
    const int tid = threadIdx.x, j = tid & 15;
    const int row = blockIdx.x * (int)(blockDim.x >> 4) + (tid >> 4);
    const bool live = row < rows;
    const int rr = live ? row : rows - 1;
    const int b = rr / Hq, h = rr % Hq, kvh = h / G, hl = h % G;
    const int64_t bkv = (int64_t)b * Hkv + kvh;
    float v[8];
    merge_row<SP, 16>(part_o, part_ml, splits_rt, bkv, hl, j, v);
    if (!out_rotated) fwht128(v, j);  // whole workgroup takes the same branch
    if (live) {
        float *orow = o + (int64_t)row * attn::D;
        *reinterpret_cast<float4 *>(orow + 4 * j) = make_float4(v[0], v[1], v[2], v[3]);
        *reinterpret_cast<float4 *>(orow + 64 + 4 * j) = make_float4(v[4], v[5], v[6], v[7]);
    }
}

// Rows that were cut into 17 .. 32 splits (one or two tokens over a long cache): 32 lanes per row, one float4 per lane
// and split, and every load of the row in flight at once.  The partials were written by workgroups all over the
// chip, so every dependent batch of loads is a round trip to memory of 2-3 us: merge_row's batches of 8 or 16 cost
// four of them here, this kernel one.  Per element the sum runs over the splits in index order with the same
// operations as merge_row: the same bits.
__global__ __launch_bounds__(64) void k_gqa_merge_wide(const float *__restrict__ part_o,
                                                       const float *__restrict__ part_ml, float *__restrict__ o,
                                                       int rows, int Hq, int Hkv, int G, int splits, int out_rotated)
{
    constexpr int SMAX = 32;
    const int tid = threadIdx.x, j = tid & 15, half = (tid >> 4) & 1;
    const int row = blockIdx.x * 2 + (tid >> 5);
    const bool live = row < rows;
    const int rr = live ? row : rows - 1;
    const int b = rr / Hq, h = rr % Hq, kvh = h / G, hl = h % G;
    const int64_t bkv = (int64_t)b * Hkv + kvh;
    const float *ml0 = part_ml + bkv * splits * 8;
    const float *po0 = part_o + (bkv * splits * 4 + hl) * attn::D + half * 64 + 4 * j;
    float ms[SMAX], ls[SMAX];
    float4 d[SMAX];
#pragma unroll
    for (int s = 0; s < SMAX; ++s) {
        const int sc = min(s, splits - 1);
        ms[s] = ml0[sc * 8 + hl];
        ls[s] = ml0[sc * 8 + 4 + hl];
        d[s] = *reinterpret_cast<const float4 *>(po0 + sc * 4 * attn::D);
    }
    float mx = -INFINITY;
#pragma unroll
    for (int s = 0; s < SMAX; ++s) mx = fmaxf(mx, ms[s]);
    float l = 0.0f, v0 = 0.0f, v1 = 0.0f, v2 = 0.0f, v3 = 0.0f;
#pragma unroll
    for (int s = 0; s < SMAX; ++s) {
        const float w = (s >= splits || ms[s] == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(ms[s] - mx);
        l = __builtin_fmaf(ls[s], w, l);
        v0 = __builtin_fmaf(d[s].x, w, v0); v1 = __builtin_fmaf(d[s].y, w, v1);
        v2 = __builtin_fmaf(d[s].z, w, v2); v3 = __builtin_fmaf(d[s].w, w, v3);
    }
    const float rl = l > 0.0f ? 1.0f / l : 0.0f;
    v0 *= rl; v1 *= rl; v2 *= rl; v3 *= rl;
    float *orow = o + (int64_t)row * attn::D;
    if (out_rotated) {
        if (live) *reinterpret_cast<float4 *>(orow + half * 64 + 4 * j) = make_float4(v0, v1, v2, v3);
        return;
    }
    // inverse rotation: the lower 16 lanes of a row collect the upper 16 lanes' elements 64 + 4j .. and run the
    // 16-lane butterfly (the upper lanes run it too, on their own values twice, and store nothing)
    const int src = (tid & ~31) | (16 + j);
    float v[8] = {v0, v1, v2, v3, __shfl(v0, src, 64), __shfl(v1, src, 64), __shfl(v2, src, 64), __shfl(v3, src, 64)};
    fwht128(v, j);
    if (live && half == 0) {
        *reinterpret_cast<float4 *>(orow + 4 * j) = make_float4(v[0], v[1], v[2], v[3]);
        *reinterpret_cast<float4 *>(orow + 64 + 4 * j) = make_float4(v[4], v[5], v[6], v[7]);
    }
}

// The merge of one token's Hq rows by one workgroup (16 lanes per head), followed by the int8 row quantizer over the
// token's Hq*128 values as they stand in the rotated basis of V: the codes and the scale are what the output
// projection's GEMV consumes when its weights were rotated along K with block 128 (x.H . (W.H)^T = x . W^T), so no
// inverse rotation and no second rotation are spent.  o_rot (optional) receives the fp32 row.
template <int SP>
__global__ __launch_bounds__(1024) void k_gqa_merge_quant(const float *__restrict__ part_o,
                                                          const float *__restrict__ part_ml,
                                                          float *__restrict__ o_rot, int8_t *__restrict__ oq,
                                                          float *__restrict__ oscale, int Hq, int Hkv, int G,
                                                          int splits_rt)
{
    __shared__ float s_max[16];
    const int tid = threadIdx.x, j = tid & 15, lane = tid & 63, wave = tid >> 6;
    const int b = blockIdx.x, h = tid >> 4;
    const int kvh = h / G, hl = h % G;
    float v[8];
    merge_row<SP>(part_o, part_ml, splits_rt, (int64_t)b * Hkv + kvh, hl, j, v);
    float a = max_lanes<16>(abs8(v));
    a = fmaxf(a, __shfl_xor(a, 16, 64));   // (a last wave may hold fewer than four heads)
    a = fmaxf(a, __shfl_xor(a, 32, 64));
    if (lane == 0) s_max[wave] = a;
    __syncthreads();
    const int nwave = (int)(blockDim.x >> 6);
    a = s_max[0];
    for (int w = 1; w < nwave; ++w) a = fmaxf(a, s_max[w]);
    const float sc = (a == 0.0f) ? 1.0f : a / 127.0f;
    const float inv = (a == 0.0f) ? 0.0f : 127.0f / a;
    const int64_t off = ((int64_t)b * Hq + h) * attn::D;
    if (tid == 0) oscale[b] = sc;
    *reinterpret_cast<uint32_t *>(oq + off + 4 * j) = quant4(v[0], v[1], v[2], v[3], inv);
    *reinterpret_cast<uint32_t *>(oq + off + 64 + 4 * j) = quant4(v[4], v[5], v[6], v[7], inv);
    if (o_rot) {
        *reinterpret_cast<float4 *>(o_rot + off + 4 * j) = make_float4(v[0], v[1], v[2], v[3]);
        *reinterpret_cast<float4 *>(o_rot + off + 64 + 4 * j) = make_float4(v[4], v[5], v[6], v[7]);
    }
}

struct SplitPlan {
    int splits, wave_tiles;
    int waves;   // of a workgroup: 4, or 8 where it sees a whole sequence
};

int max_splits(int64_t B, int64_t Hkv, int64_t T);

// Spans of 256 tokens where they are at most two workgroups a unit (and no more than 32, which the merge without codes reads at
// once, and the workspace holds), else of 704: a wave goes through all of its tiles, those past the end of its span as well, so a span that is not filled
// costs what a full one does.  us, 8 heads, before -> here (a sequence of up to 256 tokens ran in a span of 704, and few rows were cut
// into halves and quarters of 256): one sequence of 16 to 256 tokens 12.3 -> 8.9 (6.6 now that a single span needs no
// merge), of 1531 10.1 -> 9.6, 4 of 1500 13.8 -> 9.9, 32 of 256 13.3 -> 10.1, 16 of 1000 14.6 -> 14.0;
// three workgroups a unit, 32 of 700, 16.9 in spans of 256 and 15.3 in one of 704.  Past 32 spans the merge costs more than the
// units that long ones leave idle: one sequence of 8192, 8193 and 16384 tokens, 8 heads 11.1, 13.2 (21.3 in 33 spans of 256) and 15.3
// (29.3), one head 10.0, 12.7 (17.7) and 13.9 (23.5).  The merge that makes codes reads 8 spans at once (12 and 16 too) and a token in
// one workgroup: there long spans would be ahead before 32 (8192 tokens, 8 heads, 18.4, 8193 14.9; 19.3 and 25.4 before).
//
// A row of 257 to 512 tokens whose workgroup may write the output itself (`alone`) goes to one workgroup of eight waves, without a
// merge: 2 sequences of 270 tokens, 8 heads 8.4 -> 7.7 us, 16 of 384 8.8 -> 8.3, 24 of 384 11.7 -> 8.4, and the host issues one launch for
// two (9.5 -> 7.8 one after the other).  Beyond 384 tokens only from a quarter of the units on (2 of 512 would take 8.6 for 8.3;
// 0.94 to 1.00 of the time at 64 to 128 rows of 390 to 480), and beyond 480 only where two short spans a row are more than the units (0.78
// at 192 rows of 512, where the other plan's spans are long ones; 8 of 512, 8 heads 8.8 -> 9.0).
// Eight tiles a wave, up to 1024 tokens, pay where spans of 704 are two a row and the rows near the units: 24 of 900 19.3 -> 13.3, but 16 of
// 900 12.9 -> 12.7 and 8 of 900 9.2 -> 12.4.  (Not one sequence: it is cut alike with codes and without.)
static SplitPlan pick_splits(int64_t B, int64_t Hkv, int64_t T, bool alone)
{
    const int ntiles = (int)((T + 15) / 16);
    const int64_t rows = B * Hkv, cus = compute_units();
    auto spans = [&](int tiles) { return (ntiles + 4 * tiles - 1) / (4 * tiles); };
    if (alone && B > 1 && rows <= cus) {
        if (ntiles > 16 && ntiles <= 32 && (ntiles <= 24 || (ntiles <= 30 && 4 * rows >= cus) || 2 * rows > cus)) return {1, TILES_SHORT, 8};
        if (ntiles > 4 * TILES_LONG && ntiles <= 64 && 4 * rows >= 3 * cus) return {1, TILES_WIDE, 8};
    }
    const int few = spans(TILES_SHORT);
    if (few == 1 || (rows * few <= 2 * cus && few <= 32 && few <= max_splits(B, Hkv, T))) return {few, TILES_SHORT, 4};
    return {spans(TILES_LONG), TILES_LONG, 4};
}

// at least the largest split count pick_splits returns for any length in [1, T]: what workspaces are sized for
int max_splits(int64_t B, int64_t Hkv, int64_t T)
{
    const int ntiles = (int)((T + 15) / 16);
    int best = (ntiles + 4 * TILES_LONG - 1) / (4 * TILES_LONG);   // long spans: monotone in T
    if (B * Hkv < compute_units()) {
        // short spans are possible for some length: ceil(n / 16) splits (and room for 16, as there has always been)
        int s = (ntiles + 4 * TILES_SHORT - 1) / (4 * TILES_SHORT);
        if (s < 16) s = 16;
        if (s > ntiles) s = ntiles;
        if (s > best) best = s;
    }
    return best;
}

static bool merge_wide(int splits, int64_t rows) { return splits > 16 && splits <= 32 && rows <= 2 * compute_units(); }

// How many dependent batches of loads the merge of `rows` rows makes: one up to 16 splits (where it quantizes up to 8, and for 12 and
// 16) and in the kernel for 17 to 32, one per eight splits otherwise.
int merge_batches(int splits, int64_t rows, bool quant)
{
    if (splits <= (quant ? 8 : 16) || splits == 12 || splits == 16) return 1;
    return !quant && merge_wide(splits, rows) ? 1 : (splits + 7) / 8;
}

// Merge of the splits' partial results [B*Hkv, splits, 4, 128] / [B*Hkv, splits, 2, 4].  oq: one workgroup per token
// merges its Hq rows and quantizes them for the output projection (o then optionally receives the fp32 row in the
// rotated basis); otherwise 16 rows per workgroup into o.
int32_t launch_merge(const float *part_o, const float *part_ml, float *o, int8_t *oq, float *oscale, int64_t B,
                     int64_t Hq, int64_t Hkv, int splits, int out_rotated, hipStream_t s)
{
    const int G = (int)(Hq / Hkv);
    if (oq) {
#define MI_MERGEQ(SP)                                                                                           \
    launch_kernel(k_gqa_merge_quant<SP>, dim3((unsigned)B), dim3((unsigned)(Hq * 16)), 0, s, part_o, part_ml, \
                  o, oq, oscale, (int)Hq, (int)Hkv, G, splits)
        switch (splits) {
        case 1: MI_MERGEQ(1); break;
        case 2: MI_MERGEQ(2); break;
        case 3: MI_MERGEQ(3); break;
        case 4: MI_MERGEQ(4); break;
        case 5: MI_MERGEQ(5); break;
        case 6: MI_MERGEQ(6); break;
        case 7: MI_MERGEQ(-8); break;
        case 8: MI_MERGEQ(8); break;
        case 12: MI_MERGEQ(12); break;
        case 16: MI_MERGEQ(16); break;
        default: MI_MERGEQ(0); break;
        }
#undef MI_MERGEQ
        return launch_status();
    }
    const int rows = (int)(B * Hq);
    if (merge_wide(splits, rows)) {
        launch_kernel(k_gqa_merge_wide, dim3((unsigned)((rows + 1) / 2)), dim3(64), 0, s, part_o, part_ml, o, rows,
                      (int)Hq, (int)Hkv, G, splits, out_rotated);
        return launch_status();
    }
    int rpw = 16;   // rows per workgroup: fewer while that still adds workgroups below half a chip's worth
    while (rpw > 1 && rows / rpw < compute_units() / 2) rpw >>= 1;
    const dim3 mgrid((unsigned)((rows + rpw - 1) / rpw)), mblock((unsigned)(16 * rpw));
#define MI_MERGE(SP)                                                                                              \
    launch_kernel(k_gqa_merge<SP>, mgrid, mblock, 0, s, part_o, part_ml, o, rows, (int)Hq, (int)Hkv, G, \
                  splits, out_rotated)
    switch (splits) {
    case 1: MI_MERGE(1); break;
    case 2: MI_MERGE(2); break;
    case 3: MI_MERGE(3); break;
    case 4: MI_MERGE(4); break;
    case 5: MI_MERGE(5); break;
    case 6: MI_MERGE(6); break;
    case 7: MI_MERGE(-8); break;
    case 8: MI_MERGE(8); break;
    case 9: case 10: case 11: MI_MERGE(-12); break;
    case 12: MI_MERGE(12); break;
    case 13: case 14: case 15: MI_MERGE(-16); break;
    case 16: MI_MERGE(16); break;
    default: MI_MERGE(0); break;
    }
#undef MI_MERGE
    return launch_status();
}

static int64_t align_up(int64_t v, int64_t a) { return (v + a - 1) / a * a; }

}  // namespace attn
}  // namespace mi

using namespace mi;

static int32_t check_attn(int64_t B, int64_t Hq, int64_t Hkv, int64_t D, int64_t T)
{
    if (B <= 0 || Hq <= 0 || Hkv <= 0 || T <= 0) return MI_EINVAL;
    if (D != attn::D) return MI_EINVAL;
    if (Hq % Hkv || Hq / Hkv > 4) return MI_EINVAL;
    if (T > (1LL << 24) || B * Hkv > 65535) return MI_ERANGE;
    return MI_OK;
}

extern "C" int64_t mi_gqa_decode_workspace_bytes(int64_t B, int64_t Hq, int64_t Hkv, int64_t D, int64_t T)
{
    int32_t rc = check_attn(B, Hq, Hkv, D, T);
    if (rc) return rc;
    // an upper bound over every length up to T, so that a workspace sized for the capacity of a cache serves every
    // decode step: the plan is not monotone in T (a shorter sequence may be cut into more, shorter spans)
    int splits = attn::max_splits(B, Hkv, T);
    const int splits_vt = avt::max_splits(B, Hkv, T);   // one query serves both cache layouts
    if (splits_vt > splits) splits = splits_vt;
    return attn::align_up(B * Hkv * splits * 4 * attn::D * 4, 256) + attn::align_up(B * Hkv * splits * 8 * 4, 256);
}

static int32_t run_attn(const float *q, const int8_t *kq, const float *ks, const int8_t *vq, const float *vs,
                        float *o, int64_t B, int64_t Hq, int64_t Hkv, int64_t D, int64_t T, int32_t out_rotated,
                        void *workspace, int64_t workspace_bytes, int8_t *dqq, float *dsq, int32_t *ddots,
                        hipStream_t s, int64_t Tstride = 0, const int32_t *seq_len = nullptr, int8_t *oq = nullptr,
                        float *oscale = nullptr, const int32_t *block_table = nullptr, int64_t max_pages = 0,
                        int page_shift = 0)
{
    int32_t rc = check_attn(B, Hq, Hkv, D, T);
    if (rc) return rc;
    if (!q || !kq || !ks || !vq || !vs || !workspace) return MI_EINVAL;
    if (!aligned16(q) || !aligned16(kq) || !aligned16(vq) || !aligned4(ks) || !aligned4(vs) || !aligned16(workspace))
        return MI_EINVAL;
    if (workspace_bytes < mi_gqa_decode_workspace_bytes(B, Hq, Hkv, D, T)) return MI_ENOSPC;
    // (output on top of the queries: row by row, or with a merge)
    const bool alone = o && !oq && !ddots && (o == q || !overlaps(o, B * Hq * D * 4, q, B * Hq * D * 4));
    const attn::SplitPlan plan = attn::pick_splits(B, Hkv, T, alone);
    const int splits = plan.splits;
    const int ntiles = (int)((T + 15) / 16);
    attn::Params p;
    p.q = q; p.kq = kq; p.ks = ks; p.vq = vq; p.vs = vs;
    p.part_o = static_cast<float *>(workspace);
    p.part_ml = reinterpret_cast<float *>(static_cast<char *>(workspace) +
                                          attn::align_up(B * Hkv * splits * 4 * attn::D * 4, 256));
    p.dump_qq = dqq; p.dump_sq = dsq; p.dump_dots = ddots;
    p.Hq = (int)Hq; p.Hkv = (int)Hkv; p.G = (int)(Hq / Hkv); p.T = (int)T;
    p.Tstride = (int)(Tstride > 0 ? Tstride : T);
    p.seq_len = seq_len;
    p.block_table = block_table; p.max_pages = (int)max_pages; p.page_shift = page_shift;
    p.tiles_per_split = (ntiles + splits - 1) / splits;
    p.score_scale = 1.4426950408889634f * 0.08838834764831845f;  // log2(e) / sqrt(128)
    const dim3 grid((unsigned)splits, (unsigned)(B * Hkv));
    // one span: its workgroup writes the output rows, with the bits that the merge of one split gives them, and no merge is launched.
    // us, 8 heads: one sequence of 64 tokens 8.4 -> 6.6, 32 of 64 8.9 -> 7.0, 32 of 600 14.2 -> 12.2.
    const bool direct = splits == 1 && alone;
    if (direct) p.part_o = o;
    p.out_rotated = out_rotated;
#define MI_SPLIT(TILES)                                                                                       \
    do {                                                                                                      \
        if (ddots) launch_kernel((attn::k_gqa_split<true, TILES, false>), grid, dim3(256), 0, s, p);          \
        else if (direct) launch_kernel((attn::k_gqa_split<false, TILES, true>), grid, dim3(256), 0, s, p);    \
        else launch_kernel((attn::k_gqa_split<false, TILES, false>), grid, dim3(256), 0, s, p);               \
    } while (0)
    if (plan.waves == 8) {
        if (plan.wave_tiles == attn::TILES_SHORT) launch_kernel((attn::k_gqa_split<false, attn::TILES_SHORT, true, 8>), grid, dim3(512), 0, s, p);
        else launch_kernel((attn::k_gqa_split<false, attn::TILES_WIDE, true, 8>), grid, dim3(512), 0, s, p);
    } else if (plan.wave_tiles == attn::TILES_LONG) MI_SPLIT(attn::TILES_LONG);
    else MI_SPLIT(attn::TILES_SHORT);
#undef MI_SPLIT
    if (direct) return launch_status();
    rc = launch_status();
    if (rc) return rc;
    if (!o && !oq) return rc;
    return attn::launch_merge(p.part_o, p.part_ml, o, oq, oscale, B, Hq, Hkv, splits, out_rotated, s);
}

extern "C" int32_t mi_gqa_decode_attn(const float *q, const int8_t *kq, const float *ks, const int8_t *vq,
                                      const float *vs, float *o, int64_t B, int64_t Hq, int64_t Hkv, int64_t D,
                                      int64_t T, int32_t out_rotated, void *workspace, int64_t workspace_bytes,
                                      void *stream)
{
    if (!o || !aligned16(o)) return MI_EINVAL;
    return run_attn(q, kq, ks, vq, vs, o, B, Hq, Hkv, D, T, out_rotated, workspace, workspace_bytes, nullptr, nullptr,
                    nullptr, as_stream(stream));
}

extern "C" int32_t mi_gqa_decode_attn_cache(const float *q, const int8_t *kq, const float *ks, const int8_t *vq,
                                            const float *vs, float *o, int64_t B, int64_t Hq, int64_t Hkv,
                                            int64_t D, int64_t T_cap, const int32_t *seq_len, int64_t T_max,
                                            int32_t out_rotated, void *workspace, int64_t workspace_bytes,
                                            void *stream)
{
    if (!o || !aligned16(o) || !seq_len || !aligned4(seq_len)) return MI_EINVAL;
    if (T_cap <= 0 || T_max <= 0 || T_max > T_cap) return MI_EINVAL;
    if (T_cap > (1LL << 24)) return MI_ERANGE;
    return run_attn(q, kq, ks, vq, vs, o, B, Hq, Hkv, D, T_max, out_rotated, workspace, workspace_bytes, nullptr,
                    nullptr, nullptr, as_stream(stream), T_cap, seq_len);
}

extern "C" int32_t mi_gqa_decode_attn_cache_quant_i8(const float *q, const int8_t *kq, const float *ks,
                                                     const int8_t *vq, const float *vs, float *o_rot, int8_t *oq,
                                                     float *oscale, int64_t B, int64_t Hq, int64_t Hkv, int64_t D,
                                                     int64_t T_cap, const int32_t *seq_len, int64_t T_max,
                                                     void *workspace, int64_t workspace_bytes, void *stream)
{
    if (!oq || !oscale || !aligned4(oq) || !aligned4(oscale) || (o_rot && !aligned16(o_rot))) return MI_EINVAL;
    if (!seq_len || !aligned4(seq_len)) return MI_EINVAL;
    if (T_cap <= 0 || T_max <= 0 || T_max > T_cap) return MI_EINVAL;
    if (T_cap > (1LL << 24) || Hq > 64) return MI_ERANGE;
    return run_attn(q, kq, ks, vq, vs, o_rot, B, Hq, Hkv, D, T_max, 1, workspace, workspace_bytes, nullptr, nullptr,
                    nullptr, as_stream(stream), T_cap, seq_len, oq, oscale);
}

extern "C" int32_t mi_gqa_decode_attn_paged(const float *q, const int8_t *kq_pool, const float *ks_pool,
                                            const int8_t *vq_pool, const float *vs_pool, float *o,
                                            const int32_t *block_table, int64_t max_pages, int64_t page_size,
                                            int64_t B, int64_t Hq, int64_t Hkv, int64_t D, const int32_t *seq_len,
                                            int64_t T_max, int32_t out_rotated, void *workspace,
                                            int64_t workspace_bytes, void *stream)
{
    if (!o || !aligned16(o) || !seq_len || !aligned4(seq_len) || !block_table || !aligned4(block_table))
        return MI_EINVAL;
    if (page_size < 16 || (page_size & (page_size - 1)) || page_size > (1 << 20)) return MI_EINVAL;
    if (T_max <= 0 || max_pages <= 0 || T_max > max_pages * page_size) return MI_EINVAL;
    if (max_pages > (1LL << 24)) return MI_ERANGE;
    int shift = 0;
    while ((1LL << shift) < page_size) ++shift;
    return run_attn(q, kq_pool, ks_pool, vq_pool, vs_pool, o, B, Hq, Hkv, D, T_max, out_rotated, workspace,
                    workspace_bytes, nullptr, nullptr, nullptr, as_stream(stream), 0, seq_len, nullptr, nullptr,
                    block_table, max_pages, shift);
}

extern "C" int32_t mi_gqa_decode_scores_i32(const float *q, const int8_t *kq, const float *ks, const int8_t *vq,
                                            const float *vs, int8_t *qq, float *sq, int32_t *dots, int64_t B,
                                            int64_t Hq, int64_t Hkv, int64_t D, int64_t T, void *workspace,
                                            int64_t workspace_bytes, void *stream)
{
    if (!qq || !sq || !dots || !aligned4(qq) || !aligned4(sq) || !aligned4(dots)) return MI_EINVAL;
    return run_attn(q, kq, ks, vq, vs, nullptr, B, Hq, Hkv, D, T, 1, workspace, workspace_bytes, qq, sq, dots,
                    as_stream(stream));
}
