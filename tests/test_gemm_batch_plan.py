"""The work list of the batched GEMM, checked on the host (no device call): every output element of every problem
is covered by a tile that lies inside its matrix, every address the kernel forms from a tile stays inside the
operands and inside the kernel's LDS areas, and the list is balanced."""
import ctypes as C
import subprocess
import sys

import numpy as np
import pytest

BM, BN = 256, 256
CFG3 = [(2048, 6144, 4096), (2048, 14336, 4096), (2048, 14336, 4096), (2048, 4096, 14336)]


def plan(mi, shapes, cus=256):
    n = len(shapes)
    mnk = (C.c_int64 * (3 * n))(*[v for s in shapes for v in s])
    cap = 64 << 20
    buf = np.empty(cap // 4, np.int32)
    per_wg = C.c_int32()
    nbytes = mi.lib.mi_gemm_batch_plan_host(mnk, n, cus, buf.ctypes.data, cap, C.byref(per_wg))
    assert nbytes > 0, nbytes
    assert nbytes == cus * per_wg.value * 16
    return buf[:nbytes // 4].reshape(cus, per_wg.value, 4)


@pytest.mark.parametrize("shapes,cus", [
    (CFG3, 256), ([(300, 272, 512)], 256), ([(256, 256, 384)], 256), ([(2048, 6144, 384)] * 8, 256),
    ([(1066, 7264, 384)], 256), ([(735, 4512, 640), (1191, 2464, 512), (780, 3264, 384)], 256),   # ragged lists that a batch holds
    ([(1000, 1008, 384), (4096, 272, 512)], 64), (CFG3, 304), ([(777, 4096, 1024)], 7),
])
def test_every_output_is_covered_once_or_with_equal_tiles(mi, shapes, cus):
    lists = plan(mi, shapes, cus)
    cover = [np.zeros((M, N), np.uint8) for M, N, K in shapes]
    for w in range(cus):
        ended = False
        for p, m0, n0, cost in lists[w]:
            if p < 0:
                ended = True
                continue
            assert not ended, "an entry behind the end mark"
            M, N, K = shapes[p]
            assert 0 <= m0 <= M - BM and 0 <= n0 <= N - BN and n0 % 16 == 0
            assert cost == K // 128 + 10
            cover[p][m0:m0 + BM, n0:n0 + BN] += 1
        assert ended, "every list ends with a mark"
    for c, (M, N, K) in zip(cover, shapes):
        assert c.min() >= 1
        # only the last row / column of tiles is moved inwards: at most four tiles meet in a corner
        assert c.max() <= 4
        tiles = -(-M // BM) * -(-N // BN)
        assert int(c.sum()) == tiles * BM * BN


def split(mi, shapes, cus=256):
    """(bytes of the stored lists, which problems run in small tiles, the small tile)"""
    n = len(shapes)
    mnk = (C.c_int64 * (3 * n))(*[v for s in shapes for v in s])
    small, tile = np.zeros(n, np.int32), np.zeros(2, np.int32)
    nbytes = mi.lib.mi_gemm_batch_split_host(mnk, n, cus, small.ctypes.data, tile.ctypes.data)
    assert nbytes >= 0, nbytes
    return nbytes, small.tolist(), tuple(tile)


def test_stored_lists_fit_the_memory_that_the_caller_was_told_to_bring(mi):
    """Where some problems run in small tiles the lists over the others are dealt anew; they are never longer than the
    lists over all problems, whose size mi_gemm_batch_plan_bytes returns."""
    rng = np.random.default_rng(23)
    kinds = set()
    batches = [
        [(1869, 1680, 7168), (1869, 272, 512), (1869, 6848, 5504), (1869, 5792, 640)],
        [(1204, 11008, 7424), (1204, 1360, 1920), (1204, 704, 14464), (1204, 624, 3328)] + [(1204, 704, 640)] * 3 +
        [(1204, 1248, 1408)],
        [(1536, 3072, 1024), (1536, 8816, 5504), (1536, 1024, 11008)],
        [(700, 14336, 4096), (700, 4096, 28672), (700, 14336, 11008)],
        CFG3,
    ]
    for _ in range(400):
        M = int(rng.integers(256, 2049))
        batches.append([(M, 16 * int(rng.integers(16, 900)), 128 * int(rng.integers(3, 113)))
                        for _ in range(int(rng.integers(1, 9)))])
    for shapes in batches:
        nbytes, small, tile = split(mi, shapes)
        assert nbytes <= plan(mi, shapes).nbytes, shapes
        assert (nbytes == 0) == all(small) and any(small) == (tile != (0, 0)), shapes
        kinds.add("all" if all(small) else "some" if any(small) else "none")
    assert kinds == {"all", "some", "none"}
    assert split(mi, CFG3) == (plan(mi, CFG3).nbytes, [0] * 4, (0, 0))


def test_planner_without_memory_returns_an_error(mi):
    """The planner's lists for a million tiles do not fit a process whose address space may not grow: MI_ENOMEM, no exception
    through the C interface."""
    code = """
import ctypes as C, resource, sys
lib = C.CDLL(sys.argv[1])
lib.mi_gemm_batch_plan_host.restype = lib.mi_gemm_batch_split_host.restype = C.c_int64
i64 = C.c_int64
mnk, pw, out = (i64 * 3)(262144, 262144, 384), C.c_int32(), (C.c_int32 * 4)()
vm = int(open('/proc/self/statm').read().split()[0]) * resource.getpagesize()
resource.setrlimit(resource.RLIMIT_AS, (vm + (4 << 20), resource.RLIM_INFINITY))
a = lib.mi_gemm_batch_plan_host(mnk, 1, 256, out, i64(16), C.byref(pw))
b = lib.mi_gemm_batch_split_host(mnk, 1, 256, out, out)
print(a, b)
"""
    r = subprocess.run([sys.executable, "-c", code, mi.LIB_PATH], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.split() == [str(mi.ENOMEM)] * 2, (r.returncode, r.stdout, r.stderr[-500:])


def test_route_of_a_single_contraction(mi):
    """0: GEMV, 1: small tiles, 2: LDS-tiled, 3: its paired form, with the tile; what the calls refuse is refused."""
    tile = np.zeros(2, np.int32)

    def r(M, N, K, cus=256):
        return mi.lib.mi_w8a8_gemm_route_host(M, N, K, cus, tile.ctypes.data), tuple(tile.tolist())

    assert r(1, 4096, 4096) == (0, (0, 0)) and r(2, 1024, 7168) == (0, (0, 0))
    assert r(16, 4096, 4096)[0] == 1 and r(1, 16, 114816)[0] == 1
    assert r(2048, 6144, 4096) == (3, (256, 192)) and r(2000, 6144, 4096) == (2, (256, 192))
    assert r(4096, 4096, 4096) == (2, (256, 256)) and r(509, 14336, 4096) == (2, (128, 256))
    # sizes that the estimates had sent to the small tiles, 1.4 to 1.5 times slower
    assert r(2741, 13008, 10240)[0] == 2 and r(764, 16064, 9856)[0] == 2 and r(3898, 9264, 7808)[0] == 2
    rng = np.random.default_rng(3)
    for _ in range(2000):
        M, N, K = int(rng.integers(1, 3000)), 16 * int(rng.integers(1, 2000)), 128 * int(rng.integers(1, 128))
        kind, (bm, bn) = r(M, N, K)
        assert kind in (0, 1, 2, 3) and (kind == 0) == (bm == 0) and (kind != 0 or M <= 4) and (kind < 2 or M > 64)
        assert kind != 3 or (M % bm == 0 and N % bn == 0)
    # three rows of tiles either way: of 96 rows they take up to 1.1 times as long where the weights are long
    assert r(273, 5232, 5120) == (1, (128, 64)) and r(270, 8288, 6656) == (1, (128, 128)) and r(259, 5008, 1024) == (1, (96, 64))
    # more rows of tiles than the small-tile kernel counts
    assert r(1 << 30, 16, 128)[0] == 2
    for bad in [(0, 16, 128), (-1, 16, 128), (1, 8, 128), (1, 16, 64), (1, 0, 128), (1, 16, 128, 0)]:
        assert r(*bad)[0] == mi.EINVAL, bad
    assert r(1, 16, 1 << 18)[0] == mi.ERANGE and r(1 << 31, 16, 128)[0] == mi.ERANGE


def test_addresses_formed_from_a_tile_stay_inside(mi):
    """Replays the kernel's address arithmetic for the first and last tile rows/columns of a problem: global byte
    offsets of the direct-to-LDS loads (wave w of eight fills blocks w + 8q: row (w + 8q) * 8 + rho of the tile,
    chunk c ^ sigma of a 128-byte K stage; the offset is formed in 32 bits), their LDS targets (two activation and three
    weight stage buffers fill the unit's 160 KB) and the loads of a lane's scales."""
    NBX, NBW = BM // 8, BN // 8          # 1 KB blocks (8 rows x 128 B) per stage
    XSTAGE, WSTAGE = NBX * 1024, NBW * 1024
    XAREA, STAGES = 2 * XSTAGE, 2 * XSTAGE + 3 * WSTAGE
    assert STAGES == 160 * 1024
    for M, N, K in [(2048, 14336, 4096), (300, 272, 512), (256, 256, 384), (2048, 4096, 14336), (1066, 7264, 384),
                    (1667, 4784, 3200)]:
        lists = plan(mi, [(M, N, K)])
        tiles = lists[lists[:, :, 0] >= 0]
        for _, m0, n0, _ in tiles[[0, -1]]:
            for w in range(8):
                for lane in range(64):
                    rho, c = lane >> 3, lane & 7
                    sigma = ((w & 1) << 2) | (rho >> 1)
                    voff = (w * 8 + rho) * K + ((c ^ sigma) << 4)
                    for kt in (0, K // 128 - 1):
                        for rows, base, nq, lds0, stage, nbuf, lo, hi in (
                                (M, m0, NBX // 8, w * 1024, XSTAGE, 2, 0, XAREA),
                                (N, n0, NBW // 8, XAREA + w * 1024, WSTAGE, 3, XAREA, STAGES)):
                            for q in range(nq):
                                off32 = voff + kt * 128 + q * 64 * K      # what the lane adds to the tile's base
                                assert 0 <= off32 < 1 << 32
                                off = base * K + off32
                                assert 0 <= off and off + 16 <= rows * K
                                for buf in range(nbuf):
                                    lds = lds0 + buf * stage + q * 8192 + 16 * lane
                                    assert lo <= lds and lds + 16 <= hi
            # a lane's scales: wave (wm, wn), lane (r, g): rows m0 + 64 wm + 16 i + r % 8 (+ 8), four columns from
            # n0 + 128 wn + 32 jp + (16 if r >= 8) + 4 g
            for w in range(8):
                wm, wn = w >> 1, w & 1
                for lane in range(64):
                    r, g = lane & 15, lane >> 4
                    for i in range(4):
                        for half in (0, 8):
                            assert 0 <= m0 + 64 * wm + 16 * i + half + (r & 7) < M
                    for jp in range(4):
                        c0 = n0 + 128 * wn + 32 * jp + (16 if r >= 8 else 0) + 4 * g
                        assert 0 <= c0 and c0 + 4 <= N


def test_cfg3_list_is_balanced(mi):
    lists = plan(mi, CFG3)
    load = np.where(lists[:, :, 0] >= 0, lists[:, :, 3], 0).sum(axis=1)
    assert load.min() > 0
    # 1,216 tiles in rounds of 256: the longest list exceeds the mean by less than a tenth
    assert load.max() <= load.mean() * 1.10, (load.max(), load.mean())
    # workgroup id mod 8 is the XCD: the XCDs' totals differ by at most one short tile per workgroup
    per_xcd = np.array([load[x::8].max() for x in range(8)])
    assert per_xcd.max() - per_xcd.min() <= 4096 // 128 + 10, per_xcd
    # all workgroups of an XCD walk the same sequence of tile lengths (a round may leave some of them out)
    for x in range(8):
        seqs = [tuple(c for p, _, _, c in lists[w] if p >= 0) for w in range(x, 256, 8)]
        longest = max(seqs, key=len)
        for s in seqs:
            it = iter(longest)
            assert all(c in it for c in s), (x, s, longest)   # s is a subsequence of the longest list
