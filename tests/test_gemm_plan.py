"""Which kernel a GEMM runs on, and what the rule promises to it, on the CPU: the plan is made on
the host and reads no matrix."""
import random
from ctypes import byref, c_int32, c_uint64

import pytest

TWO_BUFFERS, FOUR_STAGES, ANY_SHAPE = 0, 1, 2
EXACT, EDGES, UNALIGNED = 0, 1, 2
ADDRESS = 1 << 20


def plan_of(xs, M, N, K, offset=0):
    out = (c_int32 * 8)()
    xs.check(xs.halhip().HipGemmBf16PlanOf(ADDRESS + offset, ADDRESS, ADDRESS, M, N, K, out))
    return [tuple(out[i:i + 4]) for i in (0, 4) if out[i] != 0]


def tile_rows_of(xs, M, N, K, offset=0):
    """Rows of a tile, launch by launch."""
    out = (c_int32 * 4)()
    xs.check(xs.halhip().HipGemmBf16TileRowsOf(ADDRESS + offset, ADDRESS, ADDRESS, M, N, K, out))
    return [rows for rows in out[:2] if rows != 0]


@pytest.mark.parametrize("tile", [0, 64, 128, 256])
def test_a_plan_covers_the_rows_and_assumes_only_what_holds(xs, monkeypatch, tile):
    if tile != 0:
        monkeypatch.setenv("XSCHED_HIP_GEMM_TILE", str(tile))
    rng = random.Random(tile)
    for _ in range(4000):
        M, N, K = (int(2 ** rng.uniform(0, 14)) for _ in range(3))
        unit = rng.choice([1, 8, 64, 128, 256])
        M, N, K = (max(v // u * u, u) for v, u in ((M, rng.choice([1, unit])), (N, unit), (K, unit)))
        offset = rng.choice([0, 0, 0, 2, 8])
        plan = plan_of(xs, M, N, K, offset)
        aligned = offset == 0 and N % 8 == 0 and K % 8 == 0
        case = (M, N, K, offset, plan)
        assert sum(rows for rows, *_ in plan) == M, case
        tiles, tile_rows = 0, tile_rows_of(xs, M, N, K, offset)
        assert len(tile_rows) == len(plan), case
        for (rows, edge, kernel, fit), height in zip(plan, tile_rows):
            tiles += -(-rows // height) * -(-N // edge)
            assert height == edge or (edge, kernel) == (256, TWO_BUFFERS) and height in (128, 192), case
            if kernel == ANY_SHAPE:
                assert edge == 64 and len(plan) == 1, case
                assert N < 8 or M * K < 8 or (tile == 0 and K <= 128), case
                continue
            assert N >= 8 and M * K >= 8 and (tile != 0 or K > 32 or (aligned and N % 32 == 0)), case
            assert fit == UNALIGNED or aligned, case
            assert (fit == EXACT) == (aligned and rows % height == 0 and N % edge == 0 and K % 64 == 0), case
            assert kernel == FOUR_STAGES if fit == UNALIGNED else True, case
            assert (kernel, edge) in ((TWO_BUFFERS, 256), (TWO_BUFFERS, 128), (FOUR_STAGES, 128), (FOUR_STAGES, 64)), case
            assert (kernel, edge) != (TWO_BUFFERS, 128) or fit == EXACT, case
        cmd = c_uint64()
        taken = xs.halhip().HipGemmBf16CommandCreate(byref(cmd), ADDRESS + offset, ADDRESS, ADDRESS, M, N, K, 1)
        if taken == xs.kXSchedSuccess:
            assert tiles <= 1 << 18, case
            xs.check(xs.preempt().HwCommandDestroy(cmd.value))


def test_what_large_tiles_of_fewer_rows_assume(xs):
    """Whole tiles are said of the launch's own tiles, not of square ones."""
    rng, seen = random.Random(9), set()
    for _ in range(20000):
        M, N, K = (max(unit, int(2 ** rng.uniform(8, 13)) // unit * unit) for unit in (rng.choice([64, 192, 256]), 256, 64))
        plan, heights = plan_of(xs, M, N, K), tile_rows_of(xs, M, N, K)
        for (rows, edge, kernel, fit), height in zip(plan, heights):
            assert fit == (EXACT if rows % height == 0 and N % edge == 0 else EDGES), (M, N, K, plan, heights)
            seen.add((height, fit, rows % edge == 0))
    # 192 rows: whole where 256 would not be, and ragged where 256 would be whole
    assert {(192, EXACT, False), (192, EDGES, True), (128, EDGES, False)} <= seen


@pytest.mark.parametrize("M,N,K,want", [
    # 257 to 512 tiles of 128 x 128 are two rounds for the kernel with four stages
    (1920, 2944, 704, (128, TWO_BUFFERS)), (2560, 2560, 704, (128, TWO_BUFFERS)), (2048, 2944, 2048, (128, TWO_BUFFERS)),
    # short K: a tile is little more than its first loads and its write-out
    (2048, 2944, 128, (128, TWO_BUFFERS)), (3968, 4224, 64, (128, TWO_BUFFERS)), (2944, 1792, 192, (128, TWO_BUFFERS)),
    (2048, 2048, 2048, (128, FOUR_STAGES)), (1024, 1024, 1024, (64, FOUR_STAGES)), (8192, 8192, 8192, (256, TWO_BUFFERS)),
    (4096, 4096, 4096, (256, TWO_BUFFERS)),
    # short K of ragged shapes, and where it ends
    (2000, 1999, 32, (64, ANY_SHAPE)), (4000, 4008, 32, (64, ANY_SHAPE)), (4000, 4008, 40, (256, TWO_BUFFERS)),
    (7000, 7000, 64, (64, ANY_SHAPE)), (7040, 7040, 64, (128, TWO_BUFFERS)), (7001, 7003, 128, (64, ANY_SHAPE)),
    (7001, 7003, 136, (128, FOUR_STAGES)), (4001, 4003, 48, (64, ANY_SHAPE)), (4001, 4003, 49, (128, FOUR_STAGES)),
    # rows of C of whole 64-byte pieces: only where a last round of large tiles is at most half full
    (4096, 4096, 32, (256, TWO_BUFFERS)), (8192, 8192, 24, (256, TWO_BUFFERS)), (6353, 7168, 40, (256, TWO_BUFFERS)),
    (6353, 7200, 64, (256, TWO_BUFFERS)), (1024, 1024, 32, (64, FOUR_STAGES)), (7912, 4800, 32, (64, ANY_SHAPE)),
    (7912, 4800, 40, (256, TWO_BUFFERS)), (6353, 7176, 64, (64, ANY_SHAPE)),
    (300, 301, 33, (64, FOUR_STAGES)), (8191, 515, 96, (64, ANY_SHAPE)), (2000, 1999, 64, (64, ANY_SHAPE)),
    (1000, 1001, 64, (64, FOUR_STAGES))])
def test_the_kernel_that_measured_quickest_is_taken(xs, M, N, K, want):
    assert [(edge, kernel) for _, edge, kernel, _ in plan_of(xs, M, N, K)] == [want]
