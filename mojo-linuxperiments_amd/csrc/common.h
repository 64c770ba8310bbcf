// Shared host/device helpers of libmi355_int8.so (gfx950 only).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <initializer_list>
#include <tuple>
#include <utility>

#include "../../include/mi355_int8.h"

namespace mi {

extern thread_local int32_t g_last_hip_error;

inline int32_t hip_fail(hipError_t e)
{
    g_last_hip_error = (int32_t)e;
    return MI_EIO;
}

#define MI_HIP(expr)                                     \
    do {                                                 \
        hipError_t _e = (expr);                          \
        if (_e != hipSuccess) return ::mi::hip_fail(_e); \
    } while (0)

// A launch through the call that returns its status.  The triple-bracket form returns nothing and is followed by
// hipGetLastError(), which costs 0.3 us of the 2.7 that a launch takes the host; linears of a few tokens and filling a cache are
// bound by that (kv prefill of 2048 tokens, three launches; linear of 32 tokens, two).
extern thread_local hipError_t g_launch_error;   // of the launches since the last launch_status(), the first that failed
template <typename... P, typename... A>
inline void launch_kernel(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t s, A &&...a)
{
    std::tuple<P...> args{static_cast<P>(a)...};
    const hipError_t e = std::apply(
        [&](P &...v) {
            void *at[] = {const_cast<void *>(static_cast<const void *>(&v))...};
            return hipLaunchKernel(reinterpret_cast<const void *>(kernel), grid, block, at, lds, s);
        },
        args);
    if (e != hipSuccess && g_launch_error == hipSuccess) g_launch_error = e;
}

// every kernel launch is followed by this: reports a bad launch configuration
// as MI_EIO without synchronizing
inline int32_t launch_status()
{
    if (__builtin_expect(g_launch_error == hipSuccess, 1)) return MI_OK;
    const hipError_t e = g_launch_error;
    g_launch_error = hipSuccess;
    (void)hipGetLastError();   // it is reported here and not to the caller's next check
    return hip_fail(e);
}

inline hipStream_t as_stream(void *s) { return reinterpret_cast<hipStream_t>(s); }

inline bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
inline bool aligned4(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 3u) == 0; }
// do the byte ranges [a, a + an) and [b, b + bn) share a byte (null = no range)
inline bool overlaps(const void *a, int64_t an, const void *b, int64_t bn)
{
    if (!a || !b) return false;
    const uintptr_t pa = reinterpret_cast<uintptr_t>(a), pb = reinterpret_cast<uintptr_t>(b);
    return pa < pb + (uintptr_t)bn && pb < pa + (uintptr_t)an;
}
struct Span {
    const void *at;
    int64_t bytes;
};
// does none of the ranges that a kernel writes share a byte with one that it reads, or with another that it writes: what a
// kernel needs whose workgroups all read the inputs while some already write
inline bool apart(std::initializer_list<Span> reads, std::initializer_list<Span> writes)
{
    for (auto w = writes.begin(); w != writes.end(); ++w) {
        for (const Span &r : reads)
            if (overlaps(w->at, w->bytes, r.at, r.bytes)) return false;
        for (auto v = writes.begin(); v != w; ++v)
            if (overlaps(w->at, w->bytes, v->at, v->bytes)) return false;
    }
    return true;
}

int32_t compute_units();   // of the current device, cached
int32_t lds_limit();       // largest LDS allocation of one workgroup on the current device, cached

// A kernel's dynamic-LDS limit is a setting of the (kernel, device) pair: raised once for every device that the
// kernel is launched on, and refused where the device cannot give that much.  One LdsOptIn per kernel
// instantiation (a function-local static); a race between two first launches only repeats the call.
struct LdsOptIn {
    std::atomic<uint64_t> devices{0};
};
inline int32_t lds_opt_in(LdsOptIn &st, const void *kernel, int bytes)
{
    int dev = 0;
    MI_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= 64) return MI_EINVAL;
    const uint64_t bit = 1ull << dev;
    if (st.devices.load(std::memory_order_acquire) & bit) return MI_OK;
    if (bytes > lds_limit()) return MI_ENOSPC;
    MI_HIP(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
    st.devices.fetch_or(bit, std::memory_order_release);
    return MI_OK;
}
#define MI_LDS_OPT_IN(kernel, bytes)                                                              \
    do {                                                                                          \
        static ::mi::LdsOptIn _st;                                                                \
        const int32_t _rc = ::mi::lds_opt_in(_st, reinterpret_cast<const void *>(kernel), bytes); \
        if (_rc != MI_OK) return _rc;                                                             \
    } while (0)

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int WAVE = 64;

// f(std::integral_constant<int, 0>{}), ..., f(std::integral_constant<int, N-1>{}): a loop whose index is a
// compile-time constant inside the body (register arrays indexed by it stay in registers)
template <typename F, int... Is>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, Is...>)
{
    (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F &&f)
{
    static_for_impl(static_cast<F &&>(f), std::make_integer_sequence<int, N>{});
}

}  // namespace mi
