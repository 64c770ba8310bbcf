"""GPU parity: W8A8 contraction (GEMV, small-tile and LDS-tiled matrix kernels), the
dequant epilogue and the whole rotated linear.  Gates: int32 accumulators and
int8 codes bit-exact; dequantized fp32 within rel-L2 1e-3 (in fact equal)."""
import numpy as np
import pytest

import workload

pytestmark = pytest.mark.gpu


def rand_codes(seed, shape):
    return np.random.default_rng(seed).integers(-127, 128, shape).astype(np.int8)


def gpu_gemm_i32(mi, dev, qx, qw):
    mark = dev.mark()
    dqx, dqw = dev.upload(qx), dev.upload(qw)
    dacc = dev.empty((qx.shape[0], qw.shape[0]), np.int32)
    mi.gemm_i32(dqx, dqw, dacc)
    acc = dev.download(dacc)
    dev.reset_to(mark)
    return acc


@pytest.mark.parametrize("M,N,K", [
    (1, 64, 128), (1, 6144, 4096), (4, 4096, 14336), (16, 256, 4096), (13, 48, 1024),
    (17, 64, 768), (32, 4096, 4096), (33, 128, 2048), (48, 160, 256), (64, 512, 1408),
    (2, 96, 9216), (3, 80, 11264),    # a long K for few rows, in small tiles
    # 5 to 16 tokens with thousands of rows: one to many tiles per compute unit
    (16, 6144, 4096), (5, 6144, 1024), (16, 10240, 1024), (9, 14336, 2048), (16, 14336, 4096),
    (16, 20480, 1024), (12, 24576, 1024), (16, 28672, 4096), (7, 28672, 1024),
])
def test_skinny_accumulators_bit_exact(mi, dev, orc, M, N, K):
    qx, qw = rand_codes(M * 7 + N, (M, K)), rand_codes(K + 1, (N, K))
    assert np.array_equal(gpu_gemm_i32(mi, dev, qx, qw), orc.gemm_i8_i32(qx, qw))


@pytest.mark.parametrize("M,N,K", [
    (65, 256, 128), (128, 128, 256), (256, 256, 1024), (200, 192, 512), (257, 272, 384),
    (512, 448, 768), (300, 1000 // 16 * 16, 640), (2048, 224 * 3, 512), (1024, 6144, 256),
    (4096, 4096, 256),
])
def test_tiled_accumulators_bit_exact(mi, dev, orc, M, N, K):
    qx, qw = rand_codes(M + 3 * N, (M, K)), rand_codes(K + 5, (N, K))
    assert np.array_equal(gpu_gemm_i32(mi, dev, qx, qw), orc.gemm_i8_i32(qx, qw))


@pytest.mark.parametrize("M,N,K", [
    # whole 256 x 192 and 128 x 256 tiles, one per compute unit: the kernel with two waves per SIMD.  K of 1 to 5
    # stages walks every branch of its prologue and of its last stages.
    (2048, 6144, 128), (2048, 6144, 256), (2048, 6144, 384), (2048, 6144, 512), (2048, 6144, 640),
    (2048, 4096, 128), (2048, 4096, 256), (2048, 4096, 384), (2048, 4096, 896),
])
def test_paired_wave_kernel_bit_exact(mi, dev, orc, M, N, K):
    """Every accumulator, then the dequantized form of the same product (fp32, scale by scale as the oracle does)."""
    qx, qw = rand_codes(M + N + K, (M, K)), rand_codes(K + 9, (N, K))
    want = orc.gemm_i8_i32(qx, qw)
    assert np.array_equal(gpu_gemm_i32(mi, dev, qx, qw), want)
    g = np.random.default_rng(K)
    sx = g.uniform(0.01, 1, M).astype(np.float32)
    sw = g.uniform(0.001, 0.1, N).astype(np.float32)
    mark = dev.mark()
    dy = dev.empty((M, N), np.float32)
    mi.check(mi.lib.mi_w8a8_gemm_dequant_f32(dev.upload(qx).ptr, dev.upload(sx).ptr, dev.upload(qw).ptr,
                                             dev.upload(sw).ptr, dy.ptr, M, N, K, None))
    dev.sync()
    y = dev.download(dy)
    dev.reset_to(mark)
    assert np.array_equal(y, orc.dequant(want, sx, sw))


@pytest.mark.parametrize("M,N,K,tile", [
    # the LDS-tiled kernel on a chip of 256 units, each of its tiles with rows, columns or both ragged, as few stages of K as it is
    # chosen for (its prologue and last stages branch up to 5)
    (193, 24800, 128, (128, 256)), (3200, 1968, 128, (128, 256)), (386, 12256, 256, (128, 256)),
    (193, 20784, 384, (128, 256)), (195, 20592, 512, (128, 256)), (194, 21248, 512, (128, 256)),
    (142, 27616, 640, (128, 256)), (129, 27520, 768, (128, 256)), (449, 16528, 128, (256, 192)),
    (3072, 2704, 128, (256, 192)), (324, 21984, 256, (256, 192)), (392, 16992, 384, (256, 192)),
    (387, 16496, 512, (256, 192)), (285, 24000, 512, (256, 192)), (269, 23088, 640, (256, 192)),
    (258, 23152, 768, (256, 192)), (321, 24768, 128, (256, 224)), (768, 16448, 128, (256, 224)),
    (322, 24752, 256, (256, 224)), (289, 26368, 384, (256, 224)), (266, 26416, 512, (256, 224)),
    (269, 26208, 512, (256, 224)), (258, 26400, 640, (256, 224)), (257, 26336, 768, (256, 224)),
    (3070, 16320, 640, (256, 256)), (636, 19632, 896, (256, 256)), (1280, 12848, 768, (256, 256)),
    (407, 31744, 896, (256, 256)),
])
def test_lds_tiled_kernel_ragged_bit_exact(mi, dev, orc, M, N, K, tile):
    """The shapes are chosen for the kernel that they reach: a change of the choice has to bring others."""
    got = np.zeros(2, np.int32)
    assert mi.lib.mi_w8a8_gemm_route_host(M, N, K, 256, got.ctypes.data) == 2 and tuple(got) == tile
    qx, qw = rand_codes(M + N + K, (M, K)), rand_codes(K + 17, (N, K))
    want = orc.gemm_i8_i32(qx, qw)
    assert np.array_equal(gpu_gemm_i32(mi, dev, qx, qw), want)
    g = np.random.default_rng(N)
    sx, sw = g.uniform(0.01, 1, M).astype(np.float32), g.uniform(0.001, 0.1, N).astype(np.float32)
    mark = dev.mark()
    dy = dev.empty((M, N), np.float32)
    mi.gemm_dequant(dev.upload(qx), dev.upload(sx), dev.upload(qw), dev.upload(sw), dy)
    y = dev.download(dy)
    dev.reset_to(mark)
    assert np.array_equal(y, orc.dequant(want, sx, sw))


@pytest.mark.parametrize("M,N,K", [
    # every tile of the small-tile kernel on a chip of 256 units, in its order (128 x 128 to 16 x 16): fewer stages than
    # its ring holds, a last stage that K fills in part, ragged rows and columns
    (72, 25936, 128), (692, 4752, 256), (66, 10480, 384), (809, 1360, 1024), (17, 26240, 128), (373, 4560, 128),
    (570, 992, 384), (35, 6240, 128), (258, 1568, 640), (578, 848, 128), (18, 8272, 128), (97, 2640, 384), (792, 448, 1024),
    (18, 6320, 128), (387, 544, 256), (499, 448, 128), (18, 2176, 128), (845, 80, 1664), (2, 8224, 128), (270, 624, 128),
    (61, 2080, 896), (2, 4112, 128), (7, 5872, 1536), (2, 16, 128), (9, 16, 384), (11, 2848, 512),
])
def test_small_tile_kernel_bit_exact(mi, dev, orc, M, N, K):
    qx, qw = rand_codes(M + N + K, (M, K)), rand_codes(K + 11, (N, K))
    want = orc.gemm_i8_i32(qx, qw)
    assert np.array_equal(gpu_gemm_i32(mi, dev, qx, qw), want)
    g = np.random.default_rng(M)
    sx, sw = g.uniform(0.01, 1, M).astype(np.float32), g.uniform(0.001, 0.1, N).astype(np.float32)
    mark = dev.mark()
    dy = dev.empty((M, N), np.float32)
    mi.gemm_dequant(dev.upload(qx), dev.upload(sx), dev.upload(qw), dev.upload(sw), dy)
    y = dev.download(dy)
    dev.reset_to(mark)
    assert np.array_equal(y, orc.dequant(want, sx, sw))


@pytest.mark.parametrize("M,N,K,tile", [
    # the tiles of any number of rows on a chip of 256 units, with twice as many stages as their rings hold or more, so that every
    # buffer is used again; ragged; a last stage that is whole and one that is not.  The last two: of a prompt and a chunk of it
    (195, 12352, 1280, (128, 128)), (66, 8736, 1536, (128, 64)), (34, 8240, 1280, (64, 64)), (33, 6480, 1536, (64, 32)),
    (33, 4384, 2944, (32, 48)), (33, 4528, 3072, (32, 48)), (17, 6608, 2560, (32, 32)), (17, 6576, 2432, (32, 32)),
    (17, 2304, 3072, (32, 16)), (19, 2224, 3200, (32, 16)), (7, 8432, 2432, (16, 48)), (9, 8320, 2560, (16, 48)),
    (7, 4176, 2944, (16, 32)), (9, 4112, 3072, (16, 32)), (17, 16, 3712, (16, 16)), (18, 16, 4096, (16, 16)),
    (200, 14336, 4096, (128, 128)), (509, 4096, 14336, (128, 64)),
])
def test_small_tile_kernel_past_its_ring_bit_exact(mi, dev, orc, M, N, K, tile):
    got = np.zeros(2, np.int32)
    assert mi.lib.mi_w8a8_gemm_route_host(M, N, K, 256, got.ctypes.data) == 1 and tuple(got) == tile
    test_small_tile_kernel_bit_exact(mi, dev, orc, M, N, K)


@pytest.mark.parametrize("M,N,K,tile", [
    # the tiles that 129 to 1024 rows with K from 1024 are given by the finer estimate, on a chip of 256 units: one row or 16
    # columns in the last tile, whole tiles, the fewest stages, several rounds of tiles
    (480, 9904, 1152, (160, 128)), (455, 10384, 1024, (160, 128)), (288, 7552, 2048, (96, 128)), (132, 12304, 1536, (96, 128)),
    (129, 11072, 1280, (128, 96)), (133, 10960, 1280, (128, 96)), (384, 12576, 1152, (192, 128)), (330, 13840, 1024, (192, 128)),
    (480, 3136, 1024, (96, 64)), (259, 5008, 1024, (96, 64)), (896, 1168, 1024, (64, 96)), (129, 5776, 1024, (64, 96)),
])
def test_small_tile_kernel_finer_tiles_bit_exact(mi, dev, orc, M, N, K, tile):
    got = np.zeros(2, np.int32)
    assert mi.lib.mi_w8a8_gemm_route_host(M, N, K, 256, got.ctypes.data) == 1 and tuple(got) == tile
    test_small_tile_kernel_bit_exact(mi, dev, orc, M, N, K)


def test_small_tile_kernel_more_workgroups_than_one_row_of_a_grid(mi, orc):
    """2^23 tiles of 48 columns, the last with 16: 2^32 threads, more than a grid has in one direction.  The weights repeat after a
    number of rows that shares nothing with a tile; columns around the ends of the grid's rows and others drawn are compared."""
    M, N, K, period = 5, (48 << 23) - 32, 128, 999983
    got = np.zeros(2, np.int32)
    assert mi.lib.mi_w8a8_gemm_route_host(M, N, K, 256, got.ctypes.data) == 1 and tuple(got) == (16, 48)
    big = mi.Device(arena_bytes=N * K + 4 * M * N + (1 << 20))
    try:
        qx, base = rand_codes(7, (M, K)), rand_codes(8, (period, K))
        dqx, dqw, dacc = big.upload(qx), big.empty((N, K), np.int8), big.empty((M, N), np.int32)
        mi.check(mi.lib.mi_memcpy_h2d(dqw.ptr, base.ctypes.data, base.nbytes, None))
        done = period * K
        while done < N * K:
            n = min(done, N * K - done)
            mi.check(mi.lib.mi_memcpy_d2d(dqw.ptr + done, dqw.ptr, n, None))
            done += n
        big.sync()
        mi.gemm_i32(dqx, dqw, dacc)
        want = orc.gemm_i8_i32(qx, base)
        rng = np.random.default_rng(9)
        rows = [48 * (k << 22) for k in (0, 1)] + [N]
        for at in [max(0, min(n - 2048, N - 4096)) for n in rows] + [int(v) for v in rng.integers(0, N - 4096, 60)]:
            for m in range(M):
                acc = big.download(dacc.offset(4 * (m * N + at), (4096,), np.int32))
                assert np.array_equal(acc, want[m, (at + np.arange(4096)) % period]), (m, at)
    finally:
        big.close()


@pytest.mark.parametrize("M,N,K", [
    # two to four tokens in the GEMV: its smallest and largest N and K on a chip of 256 units, four to eight chunks of K, a
    # last chunk that is not whole, rows past N in the last workgroup, three tokens in the kernel for four
    (2, 16, 3200), (2, 1280, 3968), (2, 3072, 7296), (3, 16, 5248), (4, 1536, 5376), (4, 2048, 5888),
    (2, 16, 4224), (2, 1024, 4992), (2, 1024, 5120), (2, 2048, 5504), (2, 1040, 6144), (2, 528, 7168), (2, 2048, 8064),
    (3, 16, 5504), (3, 768, 6016), (3, 1040, 7296), (4, 768, 5504), (4, 272, 6656), (4, 2048, 7296), (4, 1296, 8064),
    # one token whose waves have unequal shares of K: two, four, eight and sixteen waves a row at their fewest and most chunks,
    # a last wave with one chunk less and with one chunk in all, rows past N in the last workgroup; the first K beyond, and
    # sizes on both sides of the small tiles' share
    (1, 16, 8320), (1, 272, 11264), (1, 1040, 13312), (1, 96, 15360), (1, 48, 20608), (1, 64, 26752), (1, 32, 28672),
    (1, 112, 28800), (1, 48, 57344), (1, 32, 57472), (1, 80, 66560), (1, 16, 114688), (1, 16, 114816), (1, 3072, 8320),
    (1, 3088, 8320), (1, 10240, 8448), (1, 10256, 8448),
])
def test_gemv_of_few_tokens_bit_exact(mi, dev, orc, M, N, K):
    qx, qw = rand_codes(M + N + K, (M, K)), rand_codes(K + 13, (N, K))
    want = orc.gemm_i8_i32(qx, qw)
    assert np.array_equal(gpu_gemm_i32(mi, dev, qx, qw), want)
    g = np.random.default_rng(N)
    sx, sw = g.uniform(0.01, 1, M).astype(np.float32), g.uniform(0.001, 0.1, N).astype(np.float32)
    mark = dev.mark()
    dy = dev.empty((M, N), np.float32)
    mi.gemm_dequant(dev.upload(qx), dev.upload(sx), dev.upload(qw), dev.upload(sw), dy)
    y = dev.download(dy)
    dev.reset_to(mark)
    assert np.array_equal(y, orc.dequant(want, sx, sw))


def test_random_skinny_shapes_bit_exact(mi, dev, orc):
    """Seeded random shapes of few tokens (1 to 64, K of 1 to 39 stages, N any multiple of 16 or a multiple of 2048): the GEMV
    and the small tiles, exact against the oracle."""
    rng = np.random.default_rng(7)
    for _ in range(60):
        M, K = int(rng.integers(1, 65)), int(rng.integers(1, 40)) * 128
        N = int(rng.choice([int(rng.integers(1, 300)) * 16, 2048 * int(rng.integers(1, 15))]))
        qx = rng.integers(-127, 128, (M, K)).astype(np.int8)
        qw = rng.integers(-127, 128, (N, K)).astype(np.int8)
        assert np.array_equal(gpu_gemm_i32(mi, dev, qx, qw), orc.gemm_i8_i32(qx, qw)), (M, N, K)


def test_extreme_codes_do_not_overflow(mi, dev):
    K = 14336
    qx = np.full((80, K), 127, np.int8)
    qx[1::2] = -127
    qw = np.full((32, K), 127, np.int8)
    acc = gpu_gemm_i32(mi, dev, qx, qw)
    assert np.all(acc[0::2] == 127 * 127 * K) and np.all(acc[1::2] == -127 * 127 * K)
    acc = gpu_gemm_i32(mi, dev, qx[:16], qw)
    assert np.all(acc[0::2] == 127 * 127 * K) and np.all(acc[1::2] == -127 * 127 * K)


def test_dequant_kernel_matches_closed_form(mi, dev, orc):
    g = np.random.default_rng(3)
    acc = g.integers(-2 ** 27, 2 ** 27, (33, 80)).astype(np.int32)
    sx = g.uniform(0.01, 1, 33).astype(np.float32)
    sw = g.uniform(0.001, 0.1, 80).astype(np.float32)
    mark = dev.mark()
    dy = dev.empty(acc.shape, np.float32)
    mi.dequant(dev.upload(acc), dev.upload(sx), dev.upload(sw), dy)
    y = dev.download(dy)
    dev.reset_to(mark)
    assert np.array_equal(y, orc.dequant(acc, sx, sw))


@pytest.mark.parametrize("M,N,K", [(32, 4096, 4096), (1, 512, 4096), (16, 256, 14336), (130, 320, 1024),
                                   # one token, K <= 4096: the kernel with the quantizer inside; the rest: two kernels
                                   (1, 6144, 4096), (1, 272, 2048), (4, 6144, 4096), (2, 1024, 14336), (1, 4096, 14336)])
def test_whole_linear(mi, dev, orc, M, N, K):
    """cfg0 is the first case: x [32,4096] with outlier channels, W [4096,4096]."""
    x = workload.activations(11, M, K)
    w = workload.weights(12, N, K)
    mark = dev.mark()
    dw = dev.upload(w)
    dqw, dsw = dev.empty((N, K), np.int8), dev.empty(N, np.float32)
    mi.fwht_quant(dw, dqw, dsw, 128)                       # weight prep on the GPU
    qw, sw = dev.download(dqw), dev.download(dsw)
    qwo, swo = orc.rotate_quant_rows(w, 128)
    assert np.array_equal(qw, qwo) and np.array_equal(sw, swo)
    ws = dev.empty(mi.lib.mi_w8a8_linear_workspace_bytes(M, N, K), np.uint8)
    dy = dev.empty((M, N), np.float32)
    mi.linear(dev.upload(x), dqw, dsw, dy, 128, ws)
    y = dev.download(dy)
    qx = dev.download(ws.offset(0, (M, K), np.int8))
    dev.reset_to(mark)
    yo, qxo, sxo, acco = orc.w8a8_linear(x, qwo, swo, 128)
    assert np.array_equal(qx, qxo)
    rel = np.linalg.norm(y.astype(np.float64) - yo) / np.linalg.norm(yo.astype(np.float64))
    assert rel <= 1e-3            # the stated gate
    assert np.array_equal(y, yo)  # and in fact identical: same IEEE operations in the same order


@pytest.mark.parametrize("name,K,N", workload.PROJECTIONS)
@pytest.mark.parametrize("M", [1, 4, 16, 2048])
def test_full_size_projections(mi, dev, orc, name, K, N, M):
    """cfg1 / cfg3 shapes: sampled rows against the oracle plus a linearity
    checksum over every row: sum_n acc[m,n] == qx[m,:] . (sum_n qw[n,:])."""
    qx, qw = rand_codes(31 + M, (M, K)), rand_codes(32 + N, (N, K))
    acc = gpu_gemm_i32(mi, dev, qx, qw)
    colsum = qw.astype(np.int64).sum(axis=0)
    assert np.array_equal(acc.astype(np.int64).sum(axis=1), qx.astype(np.int64) @ colsum)
    rowsum = qx.astype(np.int64).sum(axis=0)
    assert np.array_equal(acc.astype(np.int64).sum(axis=0), qw.astype(np.int64) @ rowsum)
    rows = sorted(set([0, M - 1] + list(np.random.default_rng(M).integers(0, M, 6))))
    assert np.array_equal(acc[rows], orc.gemm_i8_i32(qx[rows], qw))


@pytest.mark.parametrize("name,K,N", [workload.PROJECTIONS[0], workload.PROJECTIONS[3]])
def test_whole_prefill_linear_end_to_end(mi, dev, orc, name, K, N):
    """cfg3, one projection per K: the whole mi_w8a8_linear_f32 at M = 2048 (rotate + quantize, tiled GEMM, dequant)
    against the oracle's linear on sampled rows (the oracle quantizes a row on its own, so a row of y depends on
    that row of x alone), and the activation codes of every row."""
    M = workload.PREFILL_M
    x = workload.activations(21, M, K)
    w = workload.weights(22, N, K)
    mark = dev.mark()
    dqw, dsw = dev.empty((N, K), np.int8), dev.empty(N, np.float32)
    keep = dev.mark()
    mi.fwht_quant(dev.upload(w), dqw, dsw, 128)
    dev.sync()
    dev.reset_to(keep)
    ws = dev.empty(mi.lib.mi_w8a8_linear_workspace_bytes(M, N, K), np.uint8)
    dy = dev.empty((M, N), np.float32)
    mi.linear(dev.upload(x), dqw, dsw, dy, 128, ws)
    y = dev.download(dy)
    qx = dev.download(ws.offset(0, (M, K), np.int8))
    qw, sw = dev.download(dqw), dev.download(dsw)
    dev.reset_to(mark)
    assert np.array_equal(qx, orc.rotate_quant_rows(x, 128)[0])
    rows = sorted(set([0, 255, 256, M - 1] + list(np.random.default_rng(K).integers(0, M, 8))))
    yo = orc.w8a8_linear(x[rows], qw, sw, 128)[0]
    assert np.linalg.norm(y[rows].astype(np.float64) - yo) <= 1e-3 * np.linalg.norm(yo.astype(np.float64))
    assert np.array_equal(y[rows], yo)
    assert np.all(np.isfinite(y))


def test_argument_errors(mi, dev):
    lib = mi.lib
    mark = dev.mark()
    b = dev.empty(1 << 16, np.int8)
    assert lib.mi_w8a8_gemm_i32(b.ptr, b.ptr, b.ptr, 4, 16, 100, None) == mi.EINVAL     # K % 128
    assert lib.mi_w8a8_gemm_i32(b.ptr, b.ptr, b.ptr, 4, 20, 128, None) == mi.EINVAL     # N % 16
    assert lib.mi_w8a8_gemm_i32(b.ptr, b.ptr + 8, b.ptr, 4, 16, 128, None) == mi.EINVAL  # alignment
    assert lib.mi_w8a8_gemm_i32(b.ptr, b.ptr, b.ptr, 4, 16, 133248, None) == mi.ERANGE  # int32 bound
    assert lib.mi_w8a8_gemm_i32(b.ptr, b.ptr, b.ptr, 0, 16, 128, None) == mi.OK
    assert lib.mi_w8a8_linear_f32(b.ptr, b.ptr, b.ptr, b.ptr, 4, 16, 128, 128, b.ptr, 16, None) == mi.ENOSPC
    dev.reset_to(mark)


@pytest.mark.parametrize("M,N,K", [
    (2, 16, 128), (2, 2064, 512), (2, 4096, 1024), (2, 6144, 4096), (2, 8208, 4096), (2, 16400, 2048), (2, 33040, 2176), (2, 41024, 3968),
    (3, 20480, 2048), (3, 20496, 2048), (4, 20496, 2176), (3, 28672, 4096), (4, 33040, 3968),
    (3, 20480, 4096), (3, 20496, 4096), (4, 20512, 4096),
])
@pytest.mark.parametrize("norm", [False, True])
def test_few_tokens_in_one_launch_are_the_two_launches(mi, dev, M, N, K, norm):
    """Rows a wave from none to many, whole chunks of K and not, both sides of the rule: y, codes, scales and the residual sum are
    those of the row kernel and the contraction, bit for bit, and nothing is written past the last token's row."""
    mark = dev.mark()
    g = np.random.default_rng(M * N + K)
    x, res = (dev.upload(g.standard_normal((M, K), dtype=np.float32)) for _ in range(2))
    gain = dev.upload(1 + 0.1 * g.standard_normal(K, dtype=np.float32))
    qw, sw = dev.upload(g.integers(-127, 128, (N, K), dtype=np.int8)), dev.upload(g.random(N, dtype=np.float32))
    poison = np.full(M + 1, np.nan, np.float32)
    y = dev.upload(np.repeat(poison[:, None], N, 1))
    h = dev.upload(np.repeat(poison[:, None], K, 1))
    xn = dev.upload(np.repeat(poison[:, None], K, 1))
    ws = dev.empty(mi.lib.mi_w8a8_linear_workspace_bytes(M, N, K), np.uint8)
    q, s, y2, h2, xn2 = dev.empty((M, K), np.int8), dev.empty(M, np.float32), dev.empty((M, N), np.float32), dev.empty((M, K), np.float32), dev.empty((M, K), np.float32)
    if norm:
        mi.check(mi.lib.mi_rmsnorm_linear_f32(x.ptr, res.ptr, gain.ptr, 1e-5, h.ptr, xn.ptr, qw.ptr, sw.ptr, y.ptr, M, N, K, 128, ws.ptr,
                                              ws.nbytes, None))
        mi.check(mi.lib.mi_rmsnorm_quant_f32_i8(x.ptr, res.ptr, gain.ptr, 1e-5, h2.ptr, xn2.ptr, q.ptr, s.ptr, M, K, 128, None))
    else:
        mi.check(mi.lib.mi_w8a8_linear_f32(x.ptr, qw.ptr, sw.ptr, y.ptr, M, N, K, 128, ws.ptr, ws.nbytes, None))
        mi.fwht_quant(x, q, s, 128)
    mi.gemm_dequant(q, s, qw, sw, y2)
    al = (M * K + 255) // 256 * 256
    assert np.array_equal(dev.download(ws.offset(0, (M, K), np.int8)), dev.download(q))
    assert np.array_equal(dev.download(ws.offset(al, (M,), np.float32)), dev.download(s))
    got = dev.download(y)
    assert np.array_equal(got[:M], dev.download(y2)) and np.isnan(got[M]).all()
    for a, b in ((h, h2), (xn, xn2)) if norm else ():
        got = dev.download(a)
        assert np.array_equal(got[:M], dev.download(b)) and np.isnan(got[M]).all()
    dev.reset_to(mark)


@pytest.mark.parametrize("M,N,K", [(2, 2064, 512), (2, 4096, 4096), (3, 20496, 4096), (4, 28672, 4096), (4, 20496, 2176)])
@pytest.mark.parametrize("norm", [False, True])
def test_few_tokens_that_are_not_all_numbers(mi, dev, M, N, K, norm):
    """One launch for several tokens: a row with an infinity, one with a NaN, one of zeros, without a residual.  Everything is as the
    row kernel and the contraction have it, and a row spoils no other."""
    mark = dev.mark()
    g = np.random.default_rng(M + N + K)
    rows = g.standard_normal((M, K), dtype=np.float32)
    rows[0, 5] = np.inf
    rows[M - 1, K - 3] = np.nan
    if M > 2:
        rows[1] = 0.0
    x, gain = dev.upload(rows), dev.upload(1 + 0.1 * g.standard_normal(K, dtype=np.float32))
    qw, sw = dev.upload(g.integers(-127, 128, (N, K), dtype=np.int8)), dev.upload(g.random(N, dtype=np.float32))
    ws = dev.empty(mi.lib.mi_w8a8_linear_workspace_bytes(M, N, K), np.uint8)
    y, y2, q, s = dev.empty((M, N), np.float32), dev.empty((M, N), np.float32), dev.empty((M, K), np.int8), dev.empty(M, np.float32)
    xn, xn2 = dev.empty((M, K), np.float32), dev.empty((M, K), np.float32)
    if norm:
        mi.check(mi.lib.mi_rmsnorm_linear_f32(x.ptr, None, gain.ptr, 1e-5, None, xn.ptr, qw.ptr, sw.ptr, y.ptr, M, N, K, 128, ws.ptr,
                                              ws.nbytes, None))
        mi.check(mi.lib.mi_rmsnorm_quant_f32_i8(x.ptr, None, gain.ptr, 1e-5, None, xn2.ptr, q.ptr, s.ptr, M, K, 128, None))
        assert np.array_equal(dev.download(xn), dev.download(xn2), equal_nan=True)
    else:
        mi.check(mi.lib.mi_w8a8_linear_f32(x.ptr, qw.ptr, sw.ptr, y.ptr, M, N, K, 128, ws.ptr, ws.nbytes, None))
        mi.fwht_quant(x, q, s, 128)
    mi.gemm_dequant(q, s, qw, sw, y2)
    al = (M * K + 255) // 256 * 256
    assert np.array_equal(dev.download(ws.offset(0, (M, K), np.int8)), dev.download(q))
    assert np.array_equal(dev.download(ws.offset(al, (M,), np.float32)), dev.download(s), equal_nan=True)
    got = dev.download(y)
    assert np.array_equal(got, dev.download(y2), equal_nan=True)
    if M > 2:
        assert np.all(got[1] == 0)
    dev.reset_to(mark)
