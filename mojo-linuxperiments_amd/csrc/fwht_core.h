// Device-side core of the block Hadamard rotation and the int8 row quantizer, shared by the stand-alone
// kernels and by the decode GEMV that quantizes its own activations.  A chunk is 8 floats of one Hadamard
// block (the two float4 at offsets 4j and BLOCK/2 + 4j, j = lane % (BLOCK/8)); the butterfly stages run in the
// fixed order h = 1, 2 (in-lane), 4 .. BLOCK/4 (across lanes), BLOCK/2 (in-lane), one fp32 add or subtract each.
#pragma once
#include "common.h"

namespace mi {

// value held by lane (lane ^ MASK); MASK in {1,2,4,8,16}
template <int MASK>
__device__ __forceinline__ float xor_lane(float v)
{
    const int i = __float_as_int(v);
    int r;
    if constexpr (MASK == 1) {
        r = __builtin_amdgcn_update_dpp(i, i, 0xB1, 0xf, 0xf, false);  // quad_perm [1,0,3,2]
    } else if constexpr (MASK == 2) {
        r = __builtin_amdgcn_update_dpp(i, i, 0x4E, 0xf, 0xf, false);  // quad_perm [2,3,0,1]
    } else {
        // ds_swizzle bit mode: lane' = ((lane & 0x1f) | 0) ^ MASK inside each half wave
        r = __builtin_amdgcn_ds_swizzle(i, 0x1F | (MASK << 10));
    }
    return __int_as_float(r);
}

// one cross-lane butterfly stage on 8 values: the lane whose MASK bit is
// clear holds x[i] and keeps x[i] + x[i+h]; its partner keeps x[i] - x[i+h]
template <int MASK>
__device__ __forceinline__ void cross_stage(float (&v)[8], unsigned negmask)
{
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float other = xor_lane<MASK>(v[e]);
        const float mine = __int_as_float(__float_as_int(v[e]) ^ negmask);  // -v on the upper lane
        v[e] = other + mine;
    }
}

// value held by lane (lane ^ MASK), MASK in {1,2,4,8}, without LDS
template <int MASK>
__device__ __forceinline__ int xor_lane_i(int v)
{
    if constexpr (MASK == 1) return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xf, 0xf, true);    // quad_perm [1,0,3,2]
    if constexpr (MASK == 2) return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xf, 0xf, true);    // quad_perm [2,3,0,1]
    if constexpr (MASK == 4)                                                              // row_half_mirror, quad_perm [3,2,1,0]
        return __builtin_amdgcn_mov_dpp(__builtin_amdgcn_mov_dpp(v, 0x141, 0xf, 0xf, true), 0x1B, 0xf, 0xf, true);
    return __builtin_amdgcn_mov_dpp(v, 0x128, 0xf, 0xf, true);                            // row_ror:8
}

template <int BLOCK>
__device__ __forceinline__ void fwht_chunk(float (&v)[8], int j)
{
    // h = 1, 2: inside each float4
#pragma unroll
    for (int b = 0; b < 8; b += 4) {
        float a0 = v[b] + v[b + 1], a1 = v[b] - v[b + 1];
        float a2 = v[b + 2] + v[b + 3], a3 = v[b + 2] - v[b + 3];
        v[b] = a0 + a2; v[b + 2] = a0 - a2;
        v[b + 1] = a1 + a3; v[b + 3] = a1 - a3;
    }
    // h = 4 .. BLOCK/4: across the lanes of the block
    cross_stage<1>(v, (j & 1) ? 0x80000000u : 0u);
    cross_stage<2>(v, (j & 2) ? 0x80000000u : 0u);
    cross_stage<4>(v, (j & 4) ? 0x80000000u : 0u);
    cross_stage<8>(v, (j & 8) ? 0x80000000u : 0u);
    if constexpr (BLOCK == 256) cross_stage<16>(v, (j & 16) ? 0x80000000u : 0u);
    // h = BLOCK/2: lower half against upper half
    constexpr float S = (BLOCK == 128) ? 0.08838834764831845f : 0.0625f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float lo = v[e] + v[e + 4], hi = v[e] - v[e + 4];
        v[e] = lo * S;
        v[e + 4] = hi * S;
    }
}

__device__ __forceinline__ float abs8(const float (&v)[8])
{
    float a = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) a = fmaxf(a, fabsf(v[e]));
    return a;
}

// The same rotation for values that only become codes: a zero may come out with the other sign, which no code and no absmax
// shows.  A decode step's row kernels have a row to a compute unit, or every unit rotates the same row, so what bounds them
// is the vector instructions of one wave (8 clocks each with one wave a SIMD).  A cross-lane stage is ONE instruction an
// element here instead of three: v += +-1 * (other lane's v) as a v_fmac whose first source comes through DPP, exact like the
// add, with no LDS swizzle (the lane xor 4 is a mirror of 8 lanes and a reversal of 4).  The upper lane of a pair is left
// with the negative of its result; the signs that this leaves are those of the lane alone and go into the last multiplication.
// In one asm block, stage by stage over the eight elements: a DPP source must have been written at least two wait states
// before, and here it was eight instructions before (s_nop for the first).
// With it the reductions below, which stay off LDS too, and quant4 and silu; us a kernel in a recorded chain of them, before ->
// now: codes of 32 rows of 4096 3.18 -> 2.46, of 16 rows of 14336 5.57 -> 3.84, of 16384 rows of 128 3.04 -> 2.61; with
// SwiGLU, 16 rows of 14336, 6.47 -> 5.30; with the norm, 16 rows of 4096, 3.43 -> 2.94 (an empty kernel takes 1.6).  Linear of one
// token, 4096 -> 6144, 7.33 -> 6.36; decode steps of 1 and 16 sequences 259.0 -> 244.0 and 390.3 -> 380.7.
template <int BLOCK>
__device__ __forceinline__ void fwht_codes(float (&v)[8], int j)
{
#pragma unroll
    for (int b = 0; b < 8; b += 4) {
        float a0 = v[b] + v[b + 1], a1 = v[b] - v[b + 1];
        float a2 = v[b + 2] + v[b + 3], a3 = v[b + 2] - v[b + 3];
        v[b] = a0 + a2; v[b + 2] = a0 - a2;
        v[b + 1] = a1 + a3; v[b + 3] = a1 - a3;
    }
    const float s1 = (j & 1) ? -1.0f : 1.0f, s2 = (j & 2) ? -1.0f : 1.0f, s4 = (j & 4) ? -1.0f : 1.0f, s8 = (j & 8) ? -1.0f : 1.0f;
    float t[8];
#define MI_EIGHT(X) X("0", "8") X("1", "9") X("2", "10") X("3", "11") X("4", "12") X("5", "13") X("6", "14") X("7", "15")
#define MI_X1(e, t) "v_fmac_f32_dpp %" e ", %" e ", %16 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
#define MI_X2(e, t) "v_fmac_f32_dpp %" e ", %" e ", %17 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
#define MI_X4A(e, t) "v_mov_b32_dpp %" t ", %" e " row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
#define MI_X4B(e, t) "v_fmac_f32_dpp %" e ", %" t ", %18 quad_perm:[3,2,1,0] row_mask:0xf bank_mask:0xf\n\t"
#define MI_X8(e, t) "v_fmac_f32_dpp %" e ", %" e ", %19 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
    asm("s_nop 1\n\t" MI_EIGHT(MI_X1) MI_EIGHT(MI_X2) MI_EIGHT(MI_X4A) MI_EIGHT(MI_X4B) MI_EIGHT(MI_X8)
        : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]), "=&v"(t[0]),
          "=&v"(t[1]), "=&v"(t[2]), "=&v"(t[3]), "=&v"(t[4]), "=&v"(t[5]), "=&v"(t[6]), "=&v"(t[7])
        : "v"(s1), "v"(s2), "v"(s4), "v"(s8));
#undef MI_EIGHT
#undef MI_X1
#undef MI_X2
#undef MI_X4A
#undef MI_X4B
#undef MI_X8
    if constexpr (BLOCK == 256) {
        // rows of 16 lanes against their neighbours, two elements at a time: a swap brings both rows of one element to the lanes
        // that add and subtract them, another brings the results home.  (With an LDS swizzle, a sign and an add an element, experts
        // of 16 tokens on the same eight of 128, whose codes the down kernel makes, took 31.0 us instead of 30.5.)
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
            const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[e]), __float_as_uint(v[e + 1]), false, false);
            const float sum = __uint_as_float(r[0]) + __uint_as_float(r[1]), dif = __uint_as_float(r[0]) - __uint_as_float(r[1]);
            const auto h = __builtin_amdgcn_permlane16_swap(__float_as_uint(sum), __float_as_uint(dif), false, false);
            v[e] = __uint_as_float(h[0]);
            v[e + 1] = __uint_as_float(h[1]);
        }
    }
    constexpr float S = (BLOCK == 128) ? 0.08838834764831845f : 0.0625f;
    const float sign = (__popc(j & 15) & 1) ? -S : S;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float lo = v[e] + v[e + 4], hi = v[e] - v[e + 4];
        v[e] = lo * sign;
        v[e + 4] = hi * sign;
    }
}

// Largest of non-negative values (never NaN: they come from fmaxf) over the 16 lanes of a row, over 32 and over the wave.
// Compared as integers, which their order allows and which needs no quieting of NaNs.
template <int CTRL>
__device__ __forceinline__ unsigned umax_dpp(unsigned a)
{
    return max(a, (unsigned)__builtin_amdgcn_mov_dpp((int)a, CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ unsigned umax16(unsigned a)
{
    a = umax_dpp<0xB1>(a);     // quad_perm [1,0,3,2]
    a = umax_dpp<0x4E>(a);     // quad_perm [2,3,0,1]
    a = umax_dpp<0x141>(a);    // row_half_mirror
    return umax_dpp<0x140>(a); // row_mirror
}
template <int LANES>
__device__ __forceinline__ float max_lanes(float v)   // every lane of the group gets the result; LANES 16, 32 or 64
{
    unsigned a = umax16(__float_as_uint(v));
    if constexpr (LANES >= 32) {
        const auto r = __builtin_amdgcn_permlane16_swap(a, a, false, false);
        a = max(r[0], r[1]);
    }
    if constexpr (LANES == 64) {
        const auto r = __builtin_amdgcn_permlane32_swap(a, a, false, false);
        a = max(r[0], r[1]);
    }
    return __uint_as_float(a);
}

// op of v and the value of lane xor OFF, which has to commute; their sum.  Both without LDS, whose shuffles are a chain of round trips
// where a wave has a SIMD to itself; us with shuffles -> here: router of 16 and 512 tokens 6.4 -> 6.2 and 12.8 -> 12.1, row-major
// attention of one sequence of 64 tokens 8.8 -> 8.4, 16 of 4096 29.9 -> 29.0, decode step of 16 with experts 239.5 -> 235.3.
template <int OFF, typename F>
__device__ __forceinline__ float with_far_lane(float v, F &&op)
{
    static_assert(OFF == 32 || OFF == 16, "");
    if constexpr (OFF == 32) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        return op(__uint_as_float(r[0]), __uint_as_float(r[1]));
    } else {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        return op(__uint_as_float(r[0]), __uint_as_float(r[1]));
    }
}
template <int OFF>
__device__ __forceinline__ float add_lane(float v)
{
    if constexpr (OFF >= 16) return with_far_lane<OFF>(v, [](float a, float b) { return a + b; });
    else return v + __int_as_float(xor_lane_i<OFF>(__float_as_int(v)));
}

// Sum of squares of a row in an order that depends on the row alone and not on how many threads share it, so that
// a kernel of 256 threads and one of 1024 produce the same bits: the eight squares of a chunk are added in element
// order, the 64 chunks of a group (chunk index / 64, one wave's worth) by a xor butterfly (every lane ends with
// the same bits, a + b being b + a), and the groups pairwise in index order (tree_sum; absent groups count as 0,
// which changes nothing).
__device__ __forceinline__ float chunk_sumsq(const float (&v)[8])
{
    float s = v[0] * v[0];
#pragma unroll
    for (int e = 1; e < 8; ++e) s += v[e] * v[e];
    return s;
}
__device__ __forceinline__ float group_sum(float s)   // lanes xor 32, 16, 8, 4, 2, 1 in this order
{
    return add_lane<1>(add_lane<2>(add_lane<4>(add_lane<8>(add_lane<16>(add_lane<32>(s))))));
}
template <int G>
__device__ __forceinline__ float tree_sum(const float *part)   // part[0 .. G-1], any G >= 1
{
    constexpr int P = G <= 1 ? 1 : 1 << (32 - __builtin_clz(G - 1));
    float t[P];
#pragma unroll
    for (int w = 0; w < P; ++w) t[w] = w < G ? part[w] : 0.0f;
#pragma unroll
    for (int n = P; n > 1; n >>= 1)
#pragma unroll
        for (int w = 0; w < n / 2; ++w) t[w] = t[2 * w] + t[2 * w + 1];
    return t[0];
}

// g / (1 + e^-g) with e^x = 2^n 2^f, n + f = x log2(e).  The steps and the two constants are those that the AMD compiler expands
// expf into (the second is its own, not the float nearest to log2(e) - 0x1.715476p+0), so that results stay what they were when expf
// was called here: compared over all floats with the expf of ROCm 7.2, the same bits.  What is relied upon is the error, at most
// 3e-7 of the result: an ulp of the exponential, half of one each of the sum and the quotient.  In place of expf's selects at the
// ends of its range, four instructions, x is clamped to where the sum no longer changes or is infinite, one.
__device__ __forceinline__ float silu(float g)
{
    const float x = -__builtin_amdgcn_fmed3f(g, -89.5f, 104.0f);
    const float hi = x * 0x1.715476p+0f;
    const float lo = __builtin_fmaf(x, 0x1.4ae0bep-26f, __builtin_fmaf(x, 0x1.715476p+0f, -hi));
    const float n = rintf(hi);
    return g / (1.0f + __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f((hi - n) + lo), (int)n));
}

// Codes of four values: clamp(rne(v * inv), -127, 127), a NaN counting as -127.  Clamped first (the bounds are whole numbers)
// and rounded by adding 1.5 * 2^23, which leaves the code in the low byte.
__device__ __forceinline__ uint32_t quant4(float a, float b, float c, float d, float inv)
{
    const uint32_t i0 = __float_as_uint(fminf(fmaxf(a * inv, -127.0f), 127.0f) + 12582912.0f);
    const uint32_t i1 = __float_as_uint(fminf(fmaxf(b * inv, -127.0f), 127.0f) + 12582912.0f);
    const uint32_t i2 = __float_as_uint(fminf(fmaxf(c * inv, -127.0f), 127.0f) + 12582912.0f);
    const uint32_t i3 = __float_as_uint(fminf(fmaxf(d * inv, -127.0f), 127.0f) + 12582912.0f);
    return __builtin_amdgcn_perm(__builtin_amdgcn_perm(i3, i2, 0x0c0c0400), __builtin_amdgcn_perm(i1, i0, 0x0c0c0400), 0x05040100);
}

}  // namespace mi
