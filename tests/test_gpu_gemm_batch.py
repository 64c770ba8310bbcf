"""GPU parity: several W8A8 contractions at once (mi_gemm_batch_*), in the kernel whose workgroups walk a list of
256 x 256 tiles, in small tiles, or some in either.  Gates: int32 accumulators bit-exact against the oracle; the dequantized form equal to the
oracle's fp32 operations; both equal, bit for bit, to the single-problem entry points."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rand_codes(seed, shape):
    return np.random.default_rng(seed).integers(-127, 128, shape).astype(np.int8)


def make_ops(dev, shapes, seed, dtype):
    """Upload codes (and scales) for every problem; returns the device operand tuples and the host arrays."""
    ops, host = [], []
    for i, (M, N, K) in enumerate(shapes):
        qx, qw = rand_codes(seed + 11 * i, (M, K)), rand_codes(seed + 11 * i + 5, (N, K))
        g = np.random.default_rng(seed + i)
        sx = g.uniform(0.01, 1, M).astype(np.float32)
        sw = g.uniform(0.001, 0.1, N).astype(np.float32)
        out = dev.empty((M, N), dtype)
        ops.append((dev.upload(qx), dev.upload(sx), dev.upload(qw), dev.upload(sw), out))
        host.append((qx, sx, qw, sw))
    return ops, host


# K of 3 to 7 stages (short tiles: the stores of the tile before them are still in flight when they end) and of 24, 25
# and 32.  The batches of fewer than about 200 tiles run in small tiles; in the others, which the list kernel walks, several
# tiles per workgroup exercise the load stream across tile boundaries, the scales that change registers' contents between
# tiles and the clearing of the accumulators, mixed K a cursor that changes its stride between tiles, and 264 rows or 1168
# columns the tiles that are moved inwards (more of those in test_batch_by_route).
@pytest.mark.parametrize("shapes", [
    [(256, 256, 384)],
    [(256, 256, 512)],
    [(300, 272, 640)],
    [(2048, 6144, 384)],
    [(2048, 6144, 896)],
    [(2048, 14336, 384)],
    [(4096, 4096, 512)],
    [(2048, 4608, 3072)],
    [(2048, 6144, 3200)],
    [(512, 384, 896), (256, 272, 384)],
    [(2048, 6144, 384), (2048, 4096, 4096), (264, 14336, 512)],
    [(1024, 1168, 768)] * 8,
])
def test_batch_accumulators_bit_exact(mi, dev, orc, shapes):
    mark = dev.mark()
    batch = mi.GemmBatch(dev, shapes)
    ops, host = make_ops(dev, shapes, 1000 + len(shapes) + shapes[0][2], np.int32)
    for o in ops:   # poison: every element must be written
        mi.check(mi.lib.mi_fill_u32(o[4].ptr, 0x7F7F7F7F, o[4].nbytes // 4, None))
    batch.run_i32([(qx, None, qw, None, out) for qx, _, qw, _, out in ops])
    dev.sync()
    for (M, N, K), o, (qx, sx, qw, sw) in zip(shapes, ops, host):
        assert np.array_equal(dev.download(o[4]), orc.gemm_i8_i32(qx, qw)), (M, N, K)
    batch.destroy()
    dev.reset_to(mark)


# batches whose list would be badly balanced: a long K in small tiles beside two round ones in a list (two launches), and
# batches that the small tiles take whole, in one launch of 128 x 64 or 128 x 128 tiles
@pytest.mark.parametrize("shapes", [
    [(509, 14336, 2048), (509, 2048, 7168), (509, 14336, 2048), (509, 3072, 2048)],
    [(300, 2048, 896), (256, 1040, 2176)],
    [(300, 3072, 2048), (300, 2048, 2048)],
    [(512, 3072, 2048), (512, 2048, 2048), (512, 2048, 5504)],
])
def test_batch_with_small_tiles(mi, dev, orc, shapes):
    mark = dev.mark()
    batch = mi.GemmBatch(dev, shapes)
    ops, host = make_ops(dev, shapes, 900 + len(shapes), np.float32)
    acc = [dev.empty((M, N), np.int32) for M, N, K in shapes]
    for b in acc + [o[4] for o in ops]:   # poison: every element must be written
        mi.check(mi.lib.mi_fill_u32(b.ptr, 0x7F7F7F7F, b.nbytes // 4, None))
    batch.run_i32([(qx, None, qw, None, a) for (qx, _, qw, _, _), a in zip(ops, acc)])
    batch.run_f32(ops)
    dev.sync()
    for o, a, (qx, sx, qw, sw) in zip(ops, acc, host):
        want = orc.gemm_i8_i32(qx, qw)
        assert np.array_equal(dev.download(a), want)
        assert np.array_equal(dev.download(o[4]), orc.dequant(want, sx, sw))
    batch.destroy()
    dev.reset_to(mark)


@pytest.mark.parametrize("shapes", [
    [(300, 2048, 896), (256, 1040, 2176)],     # in small tiles
    [(2048, 6144, 384)],                       # in the list
])
def test_batch_scales_need_four_bytes_of_alignment(mi, dev, orc, shapes):
    mark = dev.mark()
    batch = mi.GemmBatch(dev, shapes)
    ops, host = make_ops(dev, shapes, 31, np.float32)
    moved = []
    for (qx, _, qw, _, y), (_, sx, _, sw) in zip(ops, host):
        dsx, dsw = (dev.upload(np.concatenate([np.zeros(k, np.float32), v])).offset(4 * k, v.shape, np.float32)
                    for k, v in ((3, sx), (1, sw)))
        moved.append((qx, dsx, qw, dsw, y))
    batch.run_f32(moved)
    dev.sync()
    for o, (qx, sx, qw, sw) in zip(moved, host):
        assert np.array_equal(dev.download(o[4]), orc.dequant(orc.gemm_i8_i32(qx, qw), sx, sw))
    batch.destroy()
    dev.reset_to(mark)


@pytest.mark.parametrize("shapes", [
    [(256, 256, 384)],
    [(300, 272, 512)],
    [(2048, 6144, 384), (520, 4096, 1024)],
    [(2048, 6144, 4096)],
])
def test_batch_dequant_equals_the_oracle_and_the_single_call(mi, dev, orc, shapes):
    mark = dev.mark()
    batch = mi.GemmBatch(dev, shapes)
    ops, host = make_ops(dev, shapes, 77, np.float32)
    batch.run_f32(ops)
    batch.run_f32(ops)   # a second run on the same batch: nothing of the first is left behind
    dev.sync()
    for (M, N, K), (dqx, dsx, dqw, dsw, dy), (qx, sx, qw, sw) in zip(shapes, ops, host):
        y = dev.download(dy)
        assert np.array_equal(y, orc.dequant(orc.gemm_i8_i32(qx, qw), sx, sw)), (M, N, K)
        dy1 = dev.empty((M, N), np.float32)
        mi.check(mi.lib.mi_w8a8_gemm_dequant_f32(dqx.ptr, dsx.ptr, dqw.ptr, dsw.ptr, dy1.ptr, M, N, K, None))
        dev.sync()
        assert np.array_equal(y, dev.download(dy1)), (M, N, K)
    batch.destroy()
    dev.reset_to(mark)


def test_batch_full_size_projections(mi, dev, orc):
    """The four M = 2048 projections of the prefill configuration as one launch: checksums over every element
    against the single-problem kernels, sampled rows against the oracle."""
    shapes = [(2048, 6144, 4096), (2048, 14336, 4096), (2048, 14336, 4096), (2048, 4096, 14336)]
    mark = dev.mark()
    batch = mi.GemmBatch(dev, shapes)
    ops, host = make_ops(dev, shapes, 4242, np.int32)
    batch.run_i32([(qx, None, qw, None, out) for qx, _, qw, _, out in ops])
    dev.sync()
    rows = np.array([0, 1, 255, 256, 1023, 1791, 1792, 2047])
    for (M, N, K), (dqx, _, dqw, _, dacc), (qx, sx, qw, sw) in zip(shapes, ops, host):
        acc = dev.download(dacc)
        assert np.array_equal(acc[rows], orc.gemm_i8_i32(qx[rows], qw)), (M, N, K)
        m2 = dev.mark()
        dref = dev.empty((M, N), np.int32)
        mi.gemm_i32(dqx, dqw, dref)
        dev.sync()
        assert np.array_equal(acc, dev.download(dref)), (M, N, K)
        dev.reset_to(m2)
    batch.destroy()
    dev.reset_to(mark)


def test_batch_rejects_what_it_cannot_run(mi, dev):
    import ctypes as C
    i64 = C.c_int64

    def plan_bytes(shapes):
        arr = (i64 * (3 * len(shapes)))(*[v for s in shapes for v in s])
        return mi.lib.mi_gemm_batch_plan_bytes(arr, len(shapes))

    assert plan_bytes([(255, 256, 384)]) == mi.EINVAL      # fewer rows than a tile
    assert plan_bytes([(256, 240, 384)]) == mi.EINVAL      # fewer columns than a tile
    assert plan_bytes([(256, 264, 384)]) == mi.EINVAL      # N % 16
    assert plan_bytes([(256, 256, 448)]) == mi.EINVAL      # K % 128
    assert plan_bytes([(256, 256, 256)]) == mi.EINVAL      # fewer than three K stages
    assert plan_bytes([(256, 256, 384)] * 9) == mi.EINVAL  # more than eight problems
    assert plan_bytes([(256, 256, 1 << 18)]) == mi.ERANGE  # the int32 accumulator could overflow
    assert plan_bytes([(256, 256, 384)]) > 0
    mark = dev.mark()
    batch = mi.GemmBatch(dev, [(256, 256, 384)])
    qx, qw, out = dev.empty((256, 512), np.int8), dev.empty((256, 512), np.int8), dev.empty((256, 256), np.int32)
    with pytest.raises(mi.MiError) as e:   # K differs from the batch's
        batch.run_i32([(qx, None, qw, None, out)])
    assert e.value.status == mi.EINVAL
    batch.destroy()
    dev.reset_to(mark)


def test_random_batches_equal_the_single_problem_kernels(mi, dev):
    """Seeded random batches (1 to 4 problems, ragged M and N, 3 to 19 K stages, mixed K in one batch): every
    dequantized output equals, bit for bit, what the single-problem entry point writes for the same operands.  Batches as
    small as these run in small tiles, as the single problems do; test_random_batches_by_route_equal_the_oracle has the
    others, and the oracle."""
    rng = np.random.default_rng(20251125)
    for _ in range(12):
        shapes = [(int(rng.integers(256, 1200)), max(256, int(rng.integers(16, 90)) * 16), int(rng.integers(3, 20)) * 128)
                  for _ in range(int(rng.integers(1, 5)))]
        mark = dev.mark()
        ops, refs = [], []
        for M, N, K in shapes:
            qx = dev.upload(rng.integers(-127, 128, (M, K)).astype(np.int8))
            qw = dev.upload(rng.integers(-127, 128, (N, K)).astype(np.int8))
            sx = dev.upload(rng.uniform(0.01, 1, M).astype(np.float32))
            sw = dev.upload(rng.uniform(0.001, 0.1, N).astype(np.float32))
            y, ref = dev.empty((M, N), np.float32), dev.empty((M, N), np.float32)
            mi.check(mi.lib.mi_fill_u32(y.ptr, 0x7F7F7F7F, y.nbytes // 4, None))   # poison: every element must be written
            mi.check(mi.lib.mi_w8a8_gemm_dequant_f32(qx.ptr, sx.ptr, qw.ptr, sw.ptr, ref.ptr, M, N, K, None))
            ops.append((qx, sx, qw, sw, y))
            refs.append(ref)
        batch = mi.GemmBatch(dev, shapes)
        batch.run_f32(ops)
        dev.sync()
        for s, o, r in zip(shapes, ops, refs):
            assert np.array_equal(dev.download(o[4]), dev.download(r)), (shapes, s)
        batch.destroy()
        dev.reset_to(mark)


def route(mi, shapes, cus=256):
    """(which problems run in small tiles, the small tile)"""
    import ctypes as C
    mnk = (C.c_int64 * (3 * len(shapes)))(*[v for s in shapes for v in s])
    small, tile = np.zeros(len(shapes), np.int32), np.zeros(2, np.int32)
    assert mi.lib.mi_gemm_batch_split_host(mnk, len(shapes), cus, small.ctypes.data, tile.ctypes.data) >= 0
    return small.tolist(), tuple(tile.tolist())


def check_batch(mi, dev, orc, shapes, seed):
    mark = dev.mark()
    batch = mi.GemmBatch(dev, shapes)
    ops, host = make_ops(dev, shapes, seed, np.float32)
    acc = [dev.empty((M, N), np.int32) for M, N, K in shapes]
    for b in acc + [o[4] for o in ops]:   # poison: every element must be written
        mi.check(mi.lib.mi_fill_u32(b.ptr, 0x7F7F7F7F, b.nbytes // 4, None))
    batch.run_i32([(qx, None, qw, None, a) for (qx, _, qw, _, _), a in zip(ops, acc)])
    batch.run_f32(ops)
    dev.sync()
    for s, o, a, (qx, sx, qw, sw) in zip(shapes, ops, acc, host):
        want = orc.gemm_i8_i32(qx, qw)
        assert np.array_equal(dev.download(a), want), (shapes, s)
        assert np.array_equal(dev.download(o[4]), orc.dequant(want, sx, sw)), (shapes, s)
    batch.destroy()
    dev.reset_to(mark)


@pytest.mark.parametrize("shapes,small,tile", [
    # the list kernel: ragged rows, columns and both (tiles moved inwards by up to 255), K of 3, 4, 5, 7 and 25 stages, mixed
    # lengths in one list, a problem of two tiles beside one of hundreds
    ([(1066, 7264, 384)], [0], (0, 0)),
    ([(1430, 5536, 384)], [0], (0, 0)),
    ([(1667, 4784, 3200)], [0], (0, 0)),
    ([(533, 272, 896), (1029, 7616, 384)], [0, 0], (0, 0)),
    ([(1824, 2736, 384), (555, 6096, 384)], [0, 0], (0, 0)),
    ([(1124, 3792, 512), (537, 5984, 384), (1812, 608, 384)], [0, 0, 0], (0, 0)),
    ([(735, 4512, 640), (1191, 2464, 512), (780, 3264, 384)], [0, 0, 0], (0, 0)),
    # small tiles: each of the three, one problem and several
    ([(291, 5536, 384)], [1], (64, 64)),
    ([(1021, 688, 512), (667, 1888, 384)], [1, 1], (64, 64)),
    ([(300, 6128, 512), (692, 4432, 384), (792, 320, 768)], [1, 1, 1], (64, 64)),
    ([(262, 272, 384)], [1], (128, 64)),
    ([(860, 320, 1792), (302, 432, 2176), (536, 1536, 1408)], [1, 1, 1], (128, 64)),
    ([(276, 6688, 384)], [1], (128, 128)),
    ([(260, 288, 1024), (339, 6272, 512), (763, 496, 1152)], [1, 1, 1], (128, 128)),
    # some in either, each small tile
    ([(418, 4576, 384), (1137, 5856, 768), (947, 5296, 512)], [1, 0, 0], (64, 64)),
    ([(1048, 2368, 384), (564, 2752, 640), (1810, 1472, 384), (1663, 3584, 512)], [0, 1, 0, 0], (128, 64)),
    ([(875, 4272, 512), (1322, 7088, 384)], [1, 0], (128, 128)),
])
def test_batch_by_route(mi, dev, orc, shapes, small, tile):
    """Ragged batches, each chosen for the launches that it takes on 256 units: a change of the rule has to bring others."""
    assert route(mi, shapes) == (small, tile)
    check_batch(mi, dev, orc, shapes, 501 + shapes[0][0])


@pytest.mark.parametrize("shapes,small,tile", [
    # small tiles of 160 and 192 rows (K up to 8192 and more, none under 1024): one problem and several, ragged, beside the list
    ([(513, 6640, 8192)], [1], (160, 128)),
    ([(577, 5456, 1152), (388, 6544, 8192)], [1, 1], (160, 128)),
    ([(502, 8720, 1024), (803, 5360, 8192)], [0, 1], (160, 128)),
    ([(587, 4912, 1280), (675, 5152, 8192)], [1, 1], (192, 128)),
    ([(596, 6208, 8192), (376, 4480, 1280), (326, 2880, 8192)], [1, 1, 1], (192, 128)),
    ([(539, 3824, 8192), (821, 9408, 1152), (284, 8752, 8192)], [1, 0, 1], (192, 128)),
    # less than a tile of 160 or 192 rows a unit, which would take 1.2 times as long
    ([(259, 5520, 8192), (613, 3648, 1152)], [1, 1], (128, 128)),
    ([(580, 720, 1152), (265, 4704, 8192), (546, 4304, 1024)], [1, 1, 1], (128, 64)),
    ([(515, 5216, 8192), (522, 4016, 1152)], [1, 1], (128, 128)),
])
def test_batch_by_route_finer_tiles(mi, dev, orc, shapes, small, tile):
    test_batch_by_route(mi, dev, orc, shapes, small, tile)


@pytest.mark.parametrize("shapes", [
    [(783, 5008, 1664)],                                              # one tile a workgroup, moved inwards in rows and columns
    [(797, 2800, 1536), (257, 5808, 1536), (257, 2208, 1152)],
    [(595, 11088, 1024), (595, 8896, 1152)],                          # two: 8 and 9 stages, which end in either set of fragments
    [(400, 1728, 4096), (400, 6928, 1664), (400, 12560, 1152), (400, 4464, 1664)],
    [(400, 9008, 4096), (400, 5520, 1024), (400, 2000, 7168), (473, 12944, 1664)],   # up to three
    [(405, 5664, 1152), (400, 4800, 1152), (400, 7648, 4096)],        # the longest in small tiles
])
def test_batch_in_narrow_tiles(mi, dev, orc, shapes):
    """Batches whose list is of 256 x 128 tiles: its entries take half the bytes of the other list's."""
    import ctypes as C
    mnk = (C.c_int64 * (3 * len(shapes)))(*[v for s in shapes for v in s])
    small, tile, per_wg = np.zeros(len(shapes), np.int32), np.zeros(2, np.int32), C.c_int32()
    stored = mi.lib.mi_gemm_batch_split_host(mnk, len(shapes), 256, small.ctypes.data, tile.ctypes.data)
    rest = [s for s, x in zip(shapes, small) if not x]
    mnk = (C.c_int64 * (3 * len(rest)))(*[v for s in rest for v in s])
    buf = np.empty(1 << 20, np.uint8)
    assert 0 < stored != mi.lib.mi_gemm_batch_plan_host(mnk, len(rest), 256, buf.ctypes.data, buf.nbytes, C.byref(per_wg))
    check_batch(mi, dev, orc, shapes, 601 + shapes[0][0])


def test_random_batches_by_route_equal_the_oracle(mi, dev, orc):
    """Seeded random ragged batches until there are three of each kind: all in the list, all in small tiles, some in either."""
    rng = np.random.default_rng(20251203)
    seen = {"list": 0, "small": 0, "both": 0}
    while min(seen.values()) < 3:
        shapes = [(int(rng.integers(256, 2200)), int(rng.integers(17, 500)) * 16, int(rng.integers(3, 16)) * 128)
                  for _ in range(int(rng.integers(1, 6)))]
        if sum(M * N * K for M, N, K in shapes) > 1.2e10:
            continue
        small, _ = route(mi, shapes)
        kind = "small" if all(small) else "both" if any(small) else "list"
        if seen[kind] < 3:
            seen[kind] += 1
            check_batch(mi, dev, orc, shapes, 700 + sum(seen.values()))
