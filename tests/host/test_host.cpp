// Parity harness for the C++ host layer, one binary in the style of the
// upstream test program (test_linux_threading.mojo:11-16, :555-570): each test
// prints [PASS]/[FAIL]; unlike upstream, a failure also sets the exit status.
// The CPU oracle (oracle/oracle.c) is linked here as the checker only.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "../../mojo-linuxperiments_amd/host/mi355_host.hpp"

extern "C" {
int orc_rotate_quant_rows(const float *, int64_t, int64_t, int, int8_t *, float *, float *);
int orc_w8a8_linear(const float *, const int8_t *, const float *, float *, int64_t, int64_t, int64_t, int, int8_t *,
                    float *, int32_t *);
int orc_gqa_decode(const float *, const int8_t *, const float *, const int8_t *, const float *, float *, int64_t,
                   int64_t, int64_t, int64_t, int64_t, int, int8_t *, float *, int32_t *);
int orc_rmsnorm(const float *, const float *, const float *, float, float *, float *, int64_t, int64_t);
int orc_rope_rows(float *, const int32_t *, const float *, const float *, int64_t, int64_t);
int orc_swiglu(const float *, float *, int64_t, int64_t);
void orc_quant_row(const float *, int64_t, int8_t *, float *);
void orc_gemm_i8_i32(const int8_t *, const int8_t *, int32_t *, int64_t, int64_t, int64_t);
void orc_dequant(const int32_t *, const float *, const float *, float *, int64_t, int64_t);
}

using namespace mi355;

static int g_failed = 0;
static void report(const char *name, bool passed, const std::string &detail = "")
{
    std::printf("[%s] %s%s%s\n", passed ? "PASS" : "FAIL", name, detail.empty() ? "" : ": ", detail.c_str());
    if (!passed) ++g_failed;
}

// splitmix64 -> uniform -> Box-Muller: host-only synthetic inputs
struct Rng {
    uint64_t s;
    uint64_t next() { uint64_t z = (s += 0x9e3779b97f4a7c15ull); z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull; z = (z ^ (z >> 27)) * 0x94d049bb133111ebull; return z ^ (z >> 31); }
    double uni() { return ((next() >> 11) + 0.5) / 9007199254740992.0; }
    float normal() { return (float)(std::sqrt(-2.0 * std::log(uni())) * std::cos(6.283185307179586 * uni())); }
};

template <typename T>
static std::vector<T> download(const T *dev, size_t n)
{
    std::vector<T> h(n);
    mi_stream_synchronize(nullptr);
    mi_memcpy_d2h(h.data(), dev, (int64_t)(n * sizeof(T)), nullptr);
    mi_stream_synchronize(nullptr);
    return h;
}

template <typename T, typename Arena>
static T *upload(Arena &a, const std::vector<T> &h)
{
    T *d = a.template alloc<T>((int64_t)h.size());
    if (!d) return nullptr;
    mi_memcpy_h2d(d, h.data(), (int64_t)(h.size() * sizeof(T)), nullptr);
    mi_stream_synchronize(nullptr);
    return d;
}

static void test_arena(const Context &ctx)
{
    DeviceArena<256> arena(ctx, 1 << 20);
    bool ok = (bool)arena && arena.used() == 0 && arena.remaining() == (1 << 20) && arena.verify_placement();
    int *a = arena.alloc<int>(10);
    int *b = arena.alloc<int>(10);
    ok = ok && a && b && (reinterpret_cast<uintptr_t>(b) - reinterpret_cast<uintptr_t>(a)) == 256;
    const int64_t w = arena.mark();
    double *c = arena.alloc<double>(1000);
    arena.reset_to(w + 999999);  // beyond used: ignored
    ok = ok && arena.used() == w + 8000 + (256 - w % 256) % 256;
    arena.reset_to(w);
    ok = ok && arena.alloc<double>(1000) == c;
    ok = ok && arena.alloc<char>(2 << 20) == nullptr;  // exhausted: null pointer
    DeviceArena<256> moved(std::move(arena));
    ok = ok && (bool)moved && !(bool)arena && moved.verify_placement();
    moved.reset();
    ok = ok && moved.used() == 0;
    report("device_arena", ok);
}

// the pinned staging slab: same watermarks, zero-filled, and a round trip through the device
static void test_host_arena(const Context &ctx)
{
    HostArena<256> stage(ctx, 0, 2 << 20);
    bool ok = (bool)stage && stage.used() == 0 && stage.node() == 0 && stage.verify_placement();
    uint32_t *src = stage.alloc<uint32_t>(4096);
    uint32_t *dst = stage.alloc<uint32_t>(4096);
    ok = ok && src && dst && src[17] == 0 && stage.verify_placement();
    ok = ok && stage.alloc<char>(4 << 20) == nullptr;
    DeviceArena<256> arena(ctx, 1 << 20);
    uint32_t *d = arena.alloc<uint32_t>(4096);
    if (ok && d) {
        for (int i = 0; i < 4096; ++i) src[i] = 0x9e3779b9u * (uint32_t)i;
        ok = mi_memcpy_h2d(d, src, 4096 * 4, nullptr) == MI_OK && mi_memcpy_d2h(dst, d, 4096 * 4, nullptr) == MI_OK &&
             mi_stream_synchronize(nullptr) == MI_OK;
        for (int i = 0; ok && i < 4096; ++i) ok = dst[i] == src[i];
    }
    const int64_t w = stage.mark();
    (void)stage.alloc<double>(100);
    stage.reset_to(w);
    ok = ok && stage.used() == w;
    HostArena<256> moved(std::move(stage));
    ok = ok && (bool)moved && !(bool)stage;
    report("host_arena", ok);
}

static int32_t fill_op(void *stream, uint32_t *dst, uint32_t value, int64_t count)
{
    return mi_fill_u32(dst, value, count, stream);
}

static void test_stream_pool(const Context &ctx)
{
    DeviceArena<256> arena(ctx, 64 << 20);
    StreamPool pool(ctx, 4);
    bool ok = (bool)pool && pool.size() == 4;
    uint32_t *out = arena.alloc<uint32_t>(32 * 1024);
    for (int batch = 0; batch < 8 && ok; ++batch) {  // 32 launches in 8 batches of 4, output[i] == 2*i*i
        for (int i = 0; i < 4; ++i) {
            const uint32_t k = batch * 4 + i;
            ok = ok && pool.launch(fill_op, out + k * 1024, 2 * k * k, (int64_t)1024);
        }
        pool.wait_all();
    }
    std::vector<uint32_t> h = download(out, 32 * 1024);
    for (uint32_t k = 0; k < 32; ++k) ok = ok && h[k * 1024] == 2 * k * k && h[k * 1024 + 1023] == 2 * k * k;
    report("stream_pool_launch_wait_all", ok);

    // pool full -> launch returns false; wait_any frees a slot; nothing in flight -> -1
    uint32_t *big = arena.alloc<uint32_t>(8 << 20);
    int launched = 0;
    bool saw_full = false;
    // each launch is a run of fills (about a millisecond of device work), so that no slot can finish while the
    // host is still filling the pool
    auto long_fill = [&](void *s) {
        int32_t rc = MI_OK;
        for (int r = 0; r < 100 && rc == MI_OK; ++r) rc = mi_fill_u32(big, 7u, (int64_t)(8 << 20), s);
        return rc;
    };
    for (int i = 0; i < 64; ++i) {
        if (pool.launch(long_fill)) ++launched;
        else { saw_full = true; break; }
    }
    int completed = 0;
    while (pool.wait_any() >= 0) ++completed;
    report("stream_pool_full_and_wait_any", saw_full && launched == 4 && completed == 4 && pool.wait_any() == -1,
           "launched " + std::to_string(launched) + " completed " + std::to_string(completed));

    Gate gate = Gate::create(ctx);
    bool gok = gate.h && !gate.wait(pool.stream(0));  // never released
    gok = gok && pool.launch([&](void *s) { int32_t rc = mi_fill_u32(big, 9u, 1 << 20, s); gate.release(s); return rc; });
    gok = gok && pool.launch([&](void *s) { gate.wait(s); return mi_fill_u32(big, 11u, 1 << 20, s); });
    pool.wait_all();
    gok = gok && download(big, 16)[3] == 11u;
    gate.reset();
    gok = gok && !gate.wait_host();
    gate.destroy();
    report("gate_orders_streams", gok);
}

static void test_quant_linear(const Context &ctx)
{
    const int64_t M = 48, K = 1024, N = 256;
    DeviceArena<256> arena(ctx, 64 << 20);
    Rng rng{42};
    std::vector<float> x(M * K), w(N * K);
    for (auto &v : x) v = rng.normal();
    for (int64_t m = 0; m < M; ++m) x[m * K + 17] *= 20.0f;  // an outlier channel
    for (auto &v : w) v = 0.02f * rng.normal();
    float *dx = upload(arena, x), *dw = upload(arena, w);
    float *dy = arena.alloc<float>(M * N);
    QuantLinear<128> lin;
    bool ok = dx && dw && dy && lin.prepare(arena, dw, N, K, M, nullptr);
    ok = ok && lin.forward(dx, dy, M, nullptr) == MI_OK;
    ok = ok && lin.forward(dx, dy, M + 1, nullptr) == MI_ERANGE;
    std::vector<int8_t> qw = download(lin.qw, N * K), qw_ref(N * K), qx_ref(M * K);
    std::vector<float> sw = download(lin.sw, N), sw_ref(N), sx_ref(M), y = download(dy, M * N), y_ref(M * N);
    std::vector<int32_t> acc_ref(M * N);
    orc_rotate_quant_rows(w.data(), N, K, 128, qw_ref.data(), sw_ref.data(), nullptr);
    orc_w8a8_linear(x.data(), qw_ref.data(), sw_ref.data(), y_ref.data(), M, N, K, 128, qx_ref.data(), sx_ref.data(),
                    acc_ref.data());
    ok = ok && qw == qw_ref && sw == sw_ref;
    std::vector<int8_t> qx = download(static_cast<int8_t *>(lin.workspace), M * K);
    ok = ok && qx == qx_ref;
    double num = 0, den = 0;
    for (int64_t i = 0; i < M * N; ++i) { num += (double)(y[i] - y_ref[i]) * (y[i] - y_ref[i]); den += (double)y_ref[i] * y_ref[i]; }
    const double rel = std::sqrt(num / den);
    report("quant_linear_vs_oracle", ok && rel <= 1e-3, "rel-L2 " + std::to_string(rel));
}

// A prefill step through the host layer: two inputs rotated and quantized by one launch (mi_fwht_quant_batch_f32_i8),
// two contractions as a batch (GemmBatch), both against the oracle's linear on each problem: codes, scales and
// accumulators equal, outputs equal (the same fp32 operations).
static void test_gemm_batch(const Context &ctx)
{
    const int64_t M = 300, K0 = 2048, N0 = 272, K1 = 4096, N1 = 256;   // ragged in rows and columns (in small tiles)
    DeviceArena<256> arena(ctx, 128 << 20);
    Rng rng{77};
    auto gauss = [&](int64_t n, float s) { std::vector<float> v((size_t)n); for (auto &e : v) e = s * rng.normal(); return v; };
    std::vector<float> x0 = gauss(M * K0, 1.0f), x1 = gauss(M * K1, 1.0f), w0 = gauss(N0 * K0, 0.02f), w1 = gauss(N1 * K1, 0.02f);
    float *dx0 = upload(arena, x0), *dx1 = upload(arena, x1);
    QuantLinear<128> l0, l1;   // weight preparation only
    bool ok = dx0 && dx1 && l0.prepare(arena, upload(arena, w0), N0, K0, 1, nullptr) && l1.prepare(arena, upload(arena, w1), N1, K1, 1, nullptr);
    int8_t *q0 = arena.alloc<int8_t>(M * K0), *q1 = arena.alloc<int8_t>(M * K1);
    float *s0 = arena.alloc<float>(M), *s1 = arena.alloc<float>(M), *y0 = arena.alloc<float>(M * N0), *y1 = arena.alloc<float>(M * N1);
    ok = ok && q0 && q1 && s0 && s1 && y0 && y1;
    const mi_quant_rows sets[2] = {{dx0, q0, s0, M, K0}, {dx1, q1, s1, M, K1}};
    ok = ok && mi_fwht_quant_batch_f32_i8(sets, 2, 128, nullptr) == MI_OK;
    const int64_t mnk[6] = {M, N0, K0, M, N1, K1};
    GemmBatch batch;
    ok = ok && batch.prepare(arena, mnk, 2) == MI_OK && (bool)batch;
    const mi_gemm_problem p[2] = {{q0, s0, l0.qw, l0.sw, y0, M, N0, K0}, {q1, s1, l1.qw, l1.sw, y1, M, N1, K1}};
    ok = ok && batch.run(p, nullptr) == MI_OK;
    const mi_gemm_problem bad[2] = {{q0, s0, l0.qw, l0.sw, y0, M, N0, K0}, {q1, s1, l1.qw, l1.sw, y1, M, N1, K1 + 128}};
    ok = ok && batch.run(bad, nullptr) == MI_EINVAL;   // a shape that is not the batch's
    bool same = true;
    for (int i = 0; i < 2; ++i) {
        const int64_t N = i ? N1 : N0, K = i ? K1 : K0;
        const std::vector<float> &x = i ? x1 : x0, &w = i ? w1 : w0;
        std::vector<int8_t> qw_ref(N * K), qx_ref(M * K);
        std::vector<float> sw_ref(N), sx_ref(M), y_ref(M * N);
        std::vector<int32_t> acc_ref(M * N);
        orc_rotate_quant_rows(w.data(), N, K, 128, qw_ref.data(), sw_ref.data(), nullptr);
        orc_w8a8_linear(x.data(), qw_ref.data(), sw_ref.data(), y_ref.data(), M, N, K, 128, qx_ref.data(), sx_ref.data(), acc_ref.data());
        same = same && download(i ? q1 : q0, (size_t)(M * K)) == qx_ref && download(i ? s1 : s0, (size_t)M) == sx_ref &&
               download(i ? y1 : y0, (size_t)(M * N)) == y_ref;
    }
    report("gemm_batch_and_quant_batch_vs_oracle", ok && same, same ? "codes, scales and outputs equal" : "differ");
}

static void test_decode_attention(const Context &ctx)
{
    const int64_t B = 2, Hq = 8, Hkv = 2, D = 128, T = 200;
    DeviceArena<256> arena(ctx, 64 << 20);
    Rng rng{7};
    std::vector<float> q(B * Hq * D), k(B * Hkv * T * D), v(B * Hkv * T * D);
    for (auto &e : q) e = rng.normal();
    for (auto &e : k) e = rng.normal();
    for (auto &e : v) e = rng.normal();
    float *dq = upload(arena, q), *dk = upload(arena, k), *dv = upload(arena, v);
    int8_t *kq = arena.alloc<int8_t>(B * Hkv * T * D), *vq = arena.alloc<int8_t>(B * Hkv * T * D);
    float *ks = arena.alloc<float>(B * Hkv * T), *vs = arena.alloc<float>(B * Hkv * T), *o = arena.alloc<float>(B * Hq * D);
    DecodeAttention att;
    bool ok = att.prepare(arena, B, Hq, Hkv, T);
    ok = ok && DecodeAttention::quantize_rows(dk, kq, ks, B * Hkv * T, nullptr) == MI_OK;
    ok = ok && DecodeAttention::quantize_rows(dv, vq, vs, B * Hkv * T, nullptr) == MI_OK;
    ok = ok && att.forward(dq, kq, ks, vq, vs, o, false, nullptr) == MI_OK;
    std::vector<int8_t> hkq = download(kq, B * Hkv * T * D), hvq = download(vq, B * Hkv * T * D);
    std::vector<float> hks = download(ks, B * Hkv * T), hvs = download(vs, B * Hkv * T), ho = download(o, B * Hq * D);
    std::vector<float> o_ref(B * Hq * D);
    orc_gqa_decode(q.data(), hkq.data(), hks.data(), hvq.data(), hvs.data(), o_ref.data(), B, Hq, Hkv, D, T, 0, nullptr,
                   nullptr, nullptr);
    float err = 0;
    for (size_t i = 0; i < ho.size(); ++i) err = std::fmax(err, std::fabs(ho[i] - o_ref[i]));
    report("decode_attention_vs_oracle", ok && err <= 2e-3f, "max-abs " + std::to_string(err));
}

// three decode steps through KvCache: append at per-sequence positions, attend over per-sequence lengths; the
// cache rows follow the oracle quantizer bit for bit and the output follows the oracle on each sequence's prefix
// key codes of a tiled cache [rows, T_cap/16, 8 chunks, 16 tokens, 16 bytes] back in token-major order
static std::vector<int8_t> key_tiles_to_rows(const std::vector<int8_t> &kt, int64_t rows, int64_t T_cap)
{
    std::vector<int8_t> out(kt.size());
    for (int64_t r = 0; r < rows; ++r)
        for (int64_t t = 0; t < T_cap; ++t)
            for (int64_t d = 0; d < 128; ++d)
                out[(r * T_cap + t) * 128 + d] = kt[(r * T_cap + (t & ~15)) * 128 + (d >> 4) * 256 + (t & 15) * 16 + (d & 15)];
    return out;
}

static void test_kv_cache(const Context &ctx, int64_t T_cap, const char *name)
{
    const int64_t B = 2, Hq = 8, Hkv = 2, D = 128;
    DeviceArena<256> arena(ctx, 64 << 20);
    KvCache cache;
    bool ok = cache.prepare(arena, B, Hq, Hkv, T_cap, T_cap % 64 == 0) && (bool)cache;
    Rng rng{11};
    std::vector<int8_t> rkq(B * Hkv * T_cap * D, 0), rvq(B * Hkv * T_cap * D, 0);
    std::vector<float> rks(B * Hkv * T_cap, 0.0f), rvs(B * Hkv * T_cap, 0.0f);
    const int32_t start[2] = {0, 30};
    float err = 0;
    int32_t *dpos = arena.alloc<int32_t>(B), *dlen = arena.alloc<int32_t>(B);
    float *dq = arena.alloc<float>(B * Hq * D), *dk = arena.alloc<float>(B * Hkv * D), *dv = arena.alloc<float>(B * Hkv * D);
    float *dout = arena.alloc<float>(B * Hq * D);
    ok = ok && dpos && dlen && dq && dk && dv && dout;
    for (int step = 0; ok && step < 3; ++step) {
        std::vector<float> q(B * Hq * D), k(B * Hkv * D), v(B * Hkv * D);
        for (auto &e : q) e = rng.normal();
        for (auto &e : k) e = rng.normal();
        for (auto &e : v) e = rng.normal();
        // sequence 1 starts with 30 tokens the cache never received: they stay zero codes with zero scales,
        // which the oracle sees too
        int32_t pos[2] = {start[0] + step, start[1] + step}, len[2] = {pos[0] + 1, pos[1] + 1};
        mi_memcpy_h2d(dpos, pos, sizeof(pos), nullptr);
        mi_memcpy_h2d(dlen, len, sizeof(len), nullptr);
        mi_memcpy_h2d(dq, q.data(), (int64_t)q.size() * 4, nullptr);
        mi_memcpy_h2d(dk, k.data(), (int64_t)k.size() * 4, nullptr);
        mi_memcpy_h2d(dv, v.data(), (int64_t)v.size() * 4, nullptr);
        ok = ok && cache.append(dk, dv, Hkv * D, dpos, nullptr) == MI_OK;
        ok = ok && cache.attend(dq, dout, dlen, len[1], false, nullptr) == MI_OK;
        std::vector<float> o = download(dout, (size_t)(B * Hq * D));
        std::vector<int8_t> cq(B * Hkv * D), cvq(B * Hkv * D);
        std::vector<float> cs(B * Hkv), cvs(B * Hkv);
        orc_rotate_quant_rows(k.data(), B * Hkv, D, 128, cq.data(), cs.data(), nullptr);
        orc_rotate_quant_rows(v.data(), B * Hkv, D, 128, cvq.data(), cvs.data(), nullptr);
        for (int64_t b = 0; b < B; ++b)
            for (int64_t h = 0; h < Hkv; ++h) {
                const int64_t row = (b * Hkv + h) * T_cap + pos[b];
                std::copy(cq.begin() + (b * Hkv + h) * D, cq.begin() + (b * Hkv + h + 1) * D, rkq.begin() + row * D);
                std::copy(cvq.begin() + (b * Hkv + h) * D, cvq.begin() + (b * Hkv + h + 1) * D, rvq.begin() + row * D);
                rks[row] = cs[b * Hkv + h];
                rvs[row] = cvs[b * Hkv + h];
            }
        for (int64_t b = 0; b < B; ++b) {
            // the oracle takes a dense [1, Hkv, len, D] cache: gather this sequence's prefix
            const int64_t n = len[b];
            std::vector<int8_t> pk(Hkv * n * D), pv(Hkv * n * D);
            std::vector<float> pks(Hkv * n), pvs(Hkv * n), o_ref(Hq * D);
            for (int64_t h = 0; h < Hkv; ++h) {
                const int64_t row = (b * Hkv + h) * T_cap;
                std::copy(rkq.begin() + row * D, rkq.begin() + (row + n) * D, pk.begin() + h * n * D);
                std::copy(rvq.begin() + row * D, rvq.begin() + (row + n) * D, pv.begin() + h * n * D);
                std::copy(rks.begin() + row, rks.begin() + row + n, pks.begin() + h * n);
                std::copy(rvs.begin() + row, rvs.begin() + row + n, pvs.begin() + h * n);
            }
            orc_gqa_decode(q.data() + b * Hq * D, pk.data(), pks.data(), pv.data(), pvs.data(), o_ref.data(), 1, Hq, Hkv,
                           D, n, 0, nullptr, nullptr, nullptr);
            for (int64_t i = 0; i < Hq * D; ++i) err = std::fmax(err, std::fabs(o[b * Hq * D + i] - o_ref[i]));
        }
    }
    std::vector<int8_t> hkq = download(cache.kq, (size_t)(B * Hkv * T_cap * D));
    if (cache.tiled) hkq = key_tiles_to_rows(hkq, B * Hkv, T_cap);
    std::vector<float> hvs = download(cache.vs, (size_t)(B * Hkv * T_cap));
    ok = ok && hkq == rkq && hvs == rvs && cache.tiled == (T_cap % 64 == 0);
    report(name, ok && err <= 2e-3f, "max-abs " + std::to_string(err));
}

// PagedKvCache against KvCache: the same three decode steps, the paged cache under a table that hands its pages
// out in reverse; outputs must be equal bit for bit in either layout.
static void test_paged_kv_cache(const Context &ctx, bool tiled, const char *name)
{
    const int64_t B = 2, Hq = 8, Hkv = 2, D = 128, P = 64, max_pages = 3, T_cap = P * max_pages, pages = B * max_pages + 1;
    DeviceArena<256> arena(ctx, 64 << 20);
    KvCache dense;
    PagedKvCache paged;
    bool ok = dense.prepare(arena, B, Hq, Hkv, T_cap, tiled) && paged.prepare(arena, B, Hq, Hkv, pages, P, max_pages, tiled) &&
              (bool)paged && paged.tiled == tiled;
    // a cache that was never appended to must read as zero codes with zero scales in both
    ok = ok && mi_fill_u32(dense.kq, 0, B * Hkv * T_cap * D / 4, nullptr) == MI_OK &&
         mi_fill_u32(dense.vq, 0, B * Hkv * T_cap * D / 4, nullptr) == MI_OK &&
         mi_fill_u32(dense.ks, 0, B * Hkv * T_cap, nullptr) == MI_OK && mi_fill_u32(dense.vs, 0, B * Hkv * T_cap, nullptr) == MI_OK &&
         mi_fill_u32(paged.kq, 0, pages * Hkv * P * D / 4, nullptr) == MI_OK &&
         mi_fill_u32(paged.vq, 0, pages * Hkv * P * D / 4, nullptr) == MI_OK &&
         mi_fill_u32(paged.ks, 0, pages * Hkv * P, nullptr) == MI_OK && mi_fill_u32(paged.vs, 0, pages * Hkv * P, nullptr) == MI_OK;
    std::vector<int32_t> table((size_t)(B * max_pages));
    for (size_t i = 0; i < table.size(); ++i) table[i] = (int32_t)(pages - 1 - i);
    int32_t *dtable = upload(arena, table);
    Rng rng{21};
    int32_t *dpos = arena.alloc<int32_t>(B), *dlen = arena.alloc<int32_t>(B);
    float *dq = arena.alloc<float>(B * Hq * D), *dk = arena.alloc<float>(B * Hkv * D), *dv = arena.alloc<float>(B * Hkv * D);
    float *o1 = arena.alloc<float>(B * Hq * D), *o2 = arena.alloc<float>(B * Hq * D);
    ok = ok && dtable && dpos && dlen && dq && dk && dv && o1 && o2;
    const int32_t start[2] = {62, 127};   // both sequences cross a page boundary within the three steps
    bool same = true;
    for (int step = 0; ok && step < 3; ++step) {
        std::vector<float> q(B * Hq * D), k(B * Hkv * D), v(B * Hkv * D);
        for (auto &e : q) e = rng.normal();
        for (auto &e : k) e = rng.normal();
        for (auto &e : v) e = rng.normal();
        int32_t pos[2] = {start[0] + step, start[1] + step}, len[2] = {pos[0] + 1, pos[1] + 1};
        mi_memcpy_h2d(dpos, pos, sizeof(pos), nullptr);
        mi_memcpy_h2d(dlen, len, sizeof(len), nullptr);
        mi_memcpy_h2d(dq, q.data(), (int64_t)q.size() * 4, nullptr);
        mi_memcpy_h2d(dk, k.data(), (int64_t)k.size() * 4, nullptr);
        mi_memcpy_h2d(dv, v.data(), (int64_t)v.size() * 4, nullptr);
        ok = ok && dense.append(dk, dv, Hkv * D, dpos, nullptr) == MI_OK &&
             paged.append(dk, dv, Hkv * D, dtable, dpos, nullptr) == MI_OK &&
             dense.attend(dq, o1, dlen, len[1], false, nullptr) == MI_OK &&
             paged.attend(dq, o2, dtable, dlen, len[1], false, nullptr) == MI_OK;
        same = same && download(o1, (size_t)(B * Hq * D)) == download(o2, (size_t)(B * Hq * D));
    }
    // the calls that exist for tiled pages only say so for row-major ones
    const int32_t rc = paged.attend_quant(dq, o2, nullptr, nullptr, dtable, dlen, 1, nullptr);
    report(name, ok && same && (tiled || rc == MI_EINVAL), same ? "outputs equal" : "outputs differ");
}

// DecoderLayer::step against the oracle's operators chained in the same order, every stage fed what the device
// fed its next kernel (integer stages equal, fp32 stages to 2e-6 relative; attention to 2e-5 absolute)
static void test_decoder_layer(const Context &ctx)
{
    const int64_t B = 2, H = 512, Hq = 4, Hkv = 2, I = 1024, T_cap = 24, D = 128, NQ = (Hq + 2 * Hkv) * D;
    DeviceArena<256> arena(ctx, 256 << 20);
    Rng rng{3};
    auto gauss = [&](int64_t n, float s) { std::vector<float> v((size_t)n); for (auto &e : v) e = s * rng.normal(); return v; };
    std::vector<float> wqkv = gauss(NQ * H, 0.02f), wo = gauss(H * Hq * D, 0.02f), wgu = gauss(2 * I * H, 0.02f),
                       wd = gauss(H * I, 0.02f), g1 = gauss(H, 0.1f), g2 = gauss(H, 0.1f), x = gauss(B * H, 1.0f);
    for (auto &e : g1) e += 1.0f;
    for (auto &e : g2) e += 1.0f;
    std::vector<float> cs((size_t)(T_cap * 64)), sn((size_t)(T_cap * 64));
    for (int64_t t = 0; t < T_cap; ++t)
        for (int64_t i = 0; i < 64; ++i) {
            const double a = (double)t * std::pow(10000.0, -2.0 * (double)i / 128.0);
            cs[t * 64 + i] = (float)std::cos(a);
            sn[t * 64 + i] = (float)std::sin(a);
        }
    DecoderLayer layer;
    bool ok = layer.prepare(arena, B, H, Hq, Hkv, I, T_cap, T_cap % 64 == 0, upload(arena, wqkv), upload(arena, wo), upload(arena, wgu),
                            upload(arena, wd), upload(arena, g1), upload(arena, g2), upload(arena, cs), upload(arena, sn),
                            1e-5f, nullptr, true);
    const std::vector<int32_t> pos = {0, 9}, len = {1, 10};
    int32_t *dpos = upload(arena, pos), *dlen = upload(arena, len);
    float *dx = upload(arena, x), *dout = arena.alloc<float>(B * H);
    ok = ok && dpos && dlen && dx && dout && layer.step(dx, nullptr, dpos, dlen, 10, dout, nullptr) == MI_OK;
    if (!ok) { report("decoder_layer_vs_oracle", false, "set-up or launch failed"); return; }
    auto close = [](const std::vector<float> &a, const std::vector<float> &b, float tol) {
        float m = 0, d = 0;
        for (size_t i = 0; i < a.size(); ++i) { m = std::fmax(m, std::fabs(b[i])); d = std::fmax(d, std::fabs(a[i] - b[i])); }
        return d <= tol * std::fmax(m, 1.0f);
    };
    std::vector<int8_t> qw((size_t)(NQ * H)), ow((size_t)(H * Hq * D)), guw((size_t)(2 * I * H)), dw((size_t)(H * I));
    std::vector<float> qs((size_t)NQ), os((size_t)H), gus((size_t)(2 * I)), ds((size_t)H);
    orc_rotate_quant_rows(wqkv.data(), NQ, H, 128, qw.data(), qs.data(), nullptr);
    orc_rotate_quant_rows(wo.data(), H, Hq * D, 128, ow.data(), os.data(), nullptr);
    orc_rotate_quant_rows(wgu.data(), 2 * I, H, 128, guw.data(), gus.data(), nullptr);
    orc_rotate_quant_rows(wd.data(), H, I, 128, dw.data(), ds.data(), nullptr);
    std::vector<float> xn = download(layer.xn, (size_t)(B * H)), r((size_t)(B * H));
    orc_rmsnorm(x.data(), nullptr, g1.data(), 1e-5f, nullptr, r.data(), B, H);
    bool good = close(xn, r, 2e-6f);
    std::vector<float> qkv = download(layer.qkv_out, (size_t)(B * NQ)), y((size_t)(B * NQ));
    orc_w8a8_linear(xn.data(), qw.data(), qs.data(), y.data(), B, NQ, H, 128, nullptr, nullptr, nullptr);
    good = good && qkv == y;
    // rotary embedding of the query and key heads, then the cache rows of this step
    std::vector<float> q = download(layer.q, (size_t)(B * Hq * D));
    std::vector<int8_t> kq = download(layer.cache.kq, (size_t)(B * Hkv * T_cap * D)), vq = download(layer.cache.vq, (size_t)(B * Hkv * T_cap * D));
    std::vector<float> ks = download(layer.cache.ks, (size_t)(B * Hkv * T_cap)), vs = download(layer.cache.vs, (size_t)(B * Hkv * T_cap));
    for (int64_t b = 0; b < B && good; ++b) {
        std::vector<float> rows(qkv.begin() + b * NQ, qkv.begin() + b * NQ + (Hq + Hkv) * D);
        std::vector<int32_t> pp((size_t)(Hq + Hkv), pos[b]);
        orc_rope_rows(rows.data(), pp.data(), cs.data(), sn.data(), Hq + Hkv, D);
        good = good && std::equal(rows.begin(), rows.begin() + Hq * D, q.begin() + b * Hq * D);
        std::vector<int8_t> c((size_t)(Hkv * D));
        std::vector<float> sc((size_t)Hkv);
        orc_rotate_quant_rows(rows.data() + Hq * D, Hkv, D, 128, c.data(), sc.data(), nullptr);
        for (int64_t h = 0; h < Hkv; ++h) {
            const int64_t row = (b * Hkv + h) * T_cap + pos[b];
            good = good && std::equal(c.begin() + h * D, c.begin() + (h + 1) * D, kq.begin() + row * D) && ks[row] == sc[h];
        }
    }
    std::vector<float> att = download(layer.att, (size_t)(B * Hq * D));
    for (int64_t b = 0; b < B && good; ++b) {
        const int64_t n = len[b];
        std::vector<int8_t> pk((size_t)(Hkv * n * D)), pv((size_t)(Hkv * n * D));
        std::vector<float> pks((size_t)(Hkv * n)), pvs((size_t)(Hkv * n)), o_ref((size_t)(Hq * D));
        for (int64_t h = 0; h < Hkv; ++h) {
            const int64_t row = (b * Hkv + h) * T_cap;
            std::copy(kq.begin() + row * D, kq.begin() + (row + n) * D, pk.begin() + h * n * D);
            std::copy(vq.begin() + row * D, vq.begin() + (row + n) * D, pv.begin() + h * n * D);
            std::copy(ks.begin() + row, ks.begin() + row + n, pks.begin() + h * n);
            std::copy(vs.begin() + row, vs.begin() + row + n, pvs.begin() + h * n);
        }
        orc_gqa_decode(q.data() + b * Hq * D, pk.data(), pks.data(), pv.data(), pvs.data(), o_ref.data(), 1, Hq, Hkv, D, n,
                       1 /* rotated basis */, nullptr, nullptr, nullptr);
        for (int64_t i = 0; i < Hq * D; ++i) good = good && std::fabs(att[b * Hq * D + i] - o_ref[i]) <= 2e-5f;
    }
    // the output projection takes each token's attention row as it stands: one quantizer row, no rotation
    std::vector<int8_t> ca = download(layer.ca, (size_t)(B * Hq * D)), ca_ref((size_t)(B * Hq * D));
    std::vector<float> sa = download(layer.sa, (size_t)B), sa_ref((size_t)B);
    for (int64_t b = 0; b < B; ++b) orc_quant_row(att.data() + b * Hq * D, Hq * D, ca_ref.data() + b * Hq * D, &sa_ref[b]);
    good = good && ca == ca_ref && sa == sa_ref;
    std::vector<float> ao = download(layer.ao, (size_t)(B * H)), h1 = download(layer.h1, (size_t)(B * H)),
                       hn = download(layer.hn, (size_t)(B * H)), gu = download(layer.gu, (size_t)(B * 2 * I)),
                       act = download(layer.act, (size_t)(B * I)), dn = download(layer.dn, (size_t)(B * H)),
                       out = download(dout, (size_t)(B * H));
    y.assign((size_t)(B * H), 0.0f);
    {
        std::vector<int32_t> acc((size_t)(B * H));
        orc_gemm_i8_i32(ca.data(), ow.data(), acc.data(), B, H, Hq * D);
        orc_dequant(acc.data(), sa.data(), os.data(), y.data(), B, H);
    }
    good = good && ao == y;
    std::vector<float> hh((size_t)(B * H));
    orc_rmsnorm(ao.data(), x.data(), g2.data(), 1e-5f, hh.data(), r.data(), B, H);
    good = good && h1 == hh && close(hn, r, 2e-6f);
    y.assign((size_t)(B * 2 * I), 0.0f);
    orc_w8a8_linear(hn.data(), guw.data(), gus.data(), y.data(), B, 2 * I, H, 128, nullptr, nullptr, nullptr);
    good = good && gu == y;
    std::vector<float> a((size_t)(B * I));
    orc_swiglu(gu.data(), a.data(), B, I);
    good = good && close(act, a, 2e-6f);
    y.assign((size_t)(B * H), 0.0f);
    orc_w8a8_linear(act.data(), dw.data(), ds.data(), y.data(), B, H, I, 128, nullptr, nullptr, nullptr);
    good = good && dn == y;
    for (int64_t i = 0; i < B * H; ++i) good = good && out[i] == h1[i] + dn[i];
    report("decoder_layer_vs_oracle", good);
}

// Three small layers as a DecoderStack: the stack's step equals the same layers chained by hand with explicit
// residual adds between them only where the arithmetic is the same (the sum h1 + dn is formed once either way),
// and a recorded step replayed twice gives the same bits as the eager one (the caches are rewritten with the
// same rows at the same positions, so a replay is idempotent).
static void test_decoder_stack(const Context &ctx)
{
    const int64_t B = 2, H = 256, Hq = 2, Hkv = 1, I = 256, T_cap = 16, D = 128, NQ = (Hq + 2 * Hkv) * D;
    DeviceArena<256> arena(ctx, 256 << 20);
    Rng rng{11};
    auto gauss = [&](int64_t n, float s) { std::vector<float> v((size_t)n); for (auto &e : v) e = s * rng.normal(); return v; };
    std::vector<float> cs((size_t)(T_cap * 64)), sn((size_t)(T_cap * 64));
    for (int64_t t = 0; t < T_cap; ++t)
        for (int64_t i = 0; i < 64; ++i) {
            const double a = (double)t * std::pow(10000.0, -2.0 * (double)i / 128.0);
            cs[t * 64 + i] = (float)std::cos(a);
            sn[t * 64 + i] = (float)std::sin(a);
        }
    float *dcs = upload(arena, cs), *dsn = upload(arena, sn);
    DecoderStack<4> stack;
    DecoderLayer solo[3];
    bool ok = dcs && dsn;
    for (int l = 0; l < 3 && ok; ++l) {
        std::vector<float> wqkv = gauss(NQ * H, 0.05f), wo = gauss(H * Hq * D, 0.05f), wgu = gauss(2 * I * H, 0.05f),
                           wd = gauss(H * I, 0.05f), g1 = gauss(H, 0.1f), g2 = gauss(H, 0.1f);
        for (auto &e : g1) e += 1.0f;
        for (auto &e : g2) e += 1.0f;
        float *a = upload(arena, wqkv), *b = upload(arena, wo), *c = upload(arena, wgu), *d = upload(arena, wd),
              *e = upload(arena, g1), *f = upload(arena, g2);
        ok = a && b && c && d && e && f &&
             stack.add(arena, B, H, Hq, Hkv, I, T_cap, false, a, b, c, d, e, f, dcs, dsn, 1e-5f, nullptr) &&
             solo[l].prepare(arena, B, H, Hq, Hkv, I, T_cap, false, a, b, c, d, e, f, dcs, dsn, 1e-5f, nullptr);
    }
    std::vector<float> x = gauss(B * H, 1.0f);
    const std::vector<int32_t> pos = {0, 5}, len = {1, 6};
    int32_t *dpos = upload(arena, pos), *dlen = upload(arena, len);
    float *dx = upload(arena, x), *dout = arena.alloc<float>(B * H), *dref = arena.alloc<float>(B * H),
          *dmid = arena.alloc<float>(B * H);
    ok = ok && dpos && dlen && dx && dout && dref && dmid && stack.count == 3;
    const bool refuses = ok && [&] { DecoderStack<1> one; one.count = 1; return !one.add(arena, B, H, Hq, Hkv, I, T_cap, false, dx, dx, dx, dx, dx, dx, dcs, dsn, 1e-5f, nullptr); }();
    if (!ok) { report("decoder_stack", false, "set-up failed"); return; }
    // by hand: every layer closes with its own residual add, the next one starts from that sum
    bool good = solo[0].step(dx, nullptr, dpos, dlen, T_cap, dmid, nullptr) == MI_OK &&
                solo[1].step(dmid, nullptr, dpos, dlen, T_cap, dref, nullptr) == MI_OK &&
                solo[2].step(dref, nullptr, dpos, dlen, T_cap, dmid, nullptr) == MI_OK;
    const std::vector<float> want = download(dmid, (size_t)(B * H));
    good = good && stack.step(dx, dpos, dlen, T_cap, dout, nullptr) == MI_OK;
    const std::vector<float> eager = download(dout, (size_t)(B * H));
    good = good && eager == want;
    // the same step recorded and replayed
    StreamPool pool(ctx, 1);
    void *s = pool.stream(0);
    Graph g;
    good = good && g.begin(s) == MI_OK;
    const int32_t rc_step = stack.step(dx, dpos, dlen, T_cap, dout, s);
    good = (g.end(s) == MI_OK) && good && rc_step == MI_OK && (bool)g;
    for (int rep = 0; rep < 2 && good; ++rep) {
        good = mi_fill_u32(dout, 0u, B * H, s) == MI_OK && g.launch(s) == MI_OK && mi_stream_synchronize(s) == MI_OK;
        good = good && download(dout, (size_t)(B * H)) == want;
    }
    good = good && refuses && stack.step(dx, dpos, dlen, T_cap, nullptr, nullptr) == MI_EINVAL;
    report("decoder_stack", good);
}

// The decoder layer with an MoE FFN (use_moe): its FFN half is residual + RMSNorm followed by MoeFfn::forward on the
// normalized row, so the down output must equal a separate forward on that row, bit for bit, and the layer output
// the residual sum; the routing and the expert arithmetic themselves are gated against the oracle in the Python suite.
static void test_moe_decoder_layer(const Context &ctx)
{
    const int64_t B = 3, H = 512, Hq = 4, Hkv = 2, I = 256, E = 16, T_cap = 64, D = 128, NQ = (Hq + 2 * Hkv) * D;
    const int32_t topk = 2;
    DeviceArena<256> arena(ctx, 256 << 20);
    Rng rng{5};
    auto gauss = [&](int64_t n, float s) { std::vector<float> v((size_t)n); for (auto &e : v) e = s * rng.normal(); return v; };
    std::vector<float> wqkv = gauss(NQ * H, 0.02f), wo = gauss(H * Hq * D, 0.02f), g1((size_t)H, 1.0f), g2((size_t)H, 1.0f),
                       x = gauss(B * H, 1.0f), wr = gauss(E * H, 0.02f);
    std::vector<float> cs((size_t)(T_cap * 64), 1.0f), sn((size_t)(T_cap * 64), 0.0f);
    // expert weights: rotate + quantize fp32 matrices on the device
    auto prep = [&](int64_t n, int64_t k, int32_t block, int8_t *&q, float *&sc) {
        std::vector<float> w = gauss(E * n * k, 0.02f);
        float *dw = upload(arena, w);
        q = arena.alloc<int8_t>(E * n * k);
        sc = arena.alloc<float>(E * n);
        return dw && q && sc && mi_fwht_quant_f32_i8(dw, q, sc, E * n, k, block, nullptr) == MI_OK;
    };
    int8_t *wg = nullptr, *wu = nullptr, *wd = nullptr;
    float *sg = nullptr, *su = nullptr, *sd = nullptr;
    bool ok = prep(I, H, 128, wg, sg) && prep(I, H, 128, wu, su) && prep(H, I, 256, wd, sd);
    MoeFfn ffn;
    ok = ok && ffn.prepare(arena, B, H, I, E, topk);
    ffn.wr = upload(arena, wr); ffn.wg = wg; ffn.sg = sg; ffn.wu = wu; ffn.su = su; ffn.wd = wd; ffn.sd = sd;
    DecoderLayer layer;
    ok = ok && layer.prepare(arena, B, H, Hq, Hkv, I, T_cap, T_cap % 64 == 0, upload(arena, wqkv), upload(arena, wo), (const float *)nullptr,
                             (const float *)nullptr, upload(arena, g1), upload(arena, g2), upload(arena, cs),
                             upload(arena, sn), 1e-5f, nullptr);
    ok = ok && layer.use_moe(arena, ffn) && layer.cache.tiled;
    const std::vector<int32_t> pos = {0, 30, 63}, len = {1, 31, 64};
    int32_t *dpos = upload(arena, pos), *dlen = upload(arena, len);
    float *dx = upload(arena, x), *dout = arena.alloc<float>(B * H), *dy = arena.alloc<float>(B * H);
    ok = ok && dpos && dlen && dx && dout && dy && layer.step(dx, nullptr, dpos, dlen, 64, dout, nullptr) == MI_OK;
    if (!ok) { report("moe_decoder_layer", false, "set-up or launch failed"); return; }
    std::vector<float> out = download(dout, (size_t)(B * H)), h1 = download(layer.h1, (size_t)(B * H)),
                       dn = download(layer.dn, (size_t)(B * H));
    bool good = ffn.forward(layer.hn, dy, nullptr) == MI_OK && download(dy, (size_t)(B * H)) == dn;
    bool finite = true;
    for (size_t i = 0; i < out.size(); ++i) {
        good = good && out[i] == h1[i] + dn[i];
        finite = finite && std::isfinite(out[i]);
    }
    report("moe_decoder_layer", good && finite);
}

int main()
{
    Context ctx(0);
    report("context", (bool)ctx, ctx ? "CUs " + std::to_string(ctx.compute_units()) : "no gfx950 device");
    if (!ctx) return 1;
    test_arena(ctx);
    test_host_arena(ctx);
    test_stream_pool(ctx);
    test_quant_linear(ctx);
    test_gemm_batch(ctx);
    test_decode_attention(ctx);
    test_kv_cache(ctx, 40, "kv_cache_append_attend_vs_oracle");
    test_kv_cache(ctx, 64, "kv_cache_tiled_layouts_append_attend_vs_oracle");
    test_paged_kv_cache(ctx, false, "paged_kv_cache_row_major_equals_dense");
    test_paged_kv_cache(ctx, true, "paged_kv_cache_tiled_equals_dense");
    test_decoder_layer(ctx);
    test_decoder_stack(ctx);
    test_moe_decoder_layer(ctx);
    std::printf("%s\n", g_failed ? "SOME TESTS FAILED" : "ALL PASSED");
    return g_failed ? 1 : 0;
}
