"""Products whose rows lie off 16-byte boundaries and are copied to rows on them first: when that is
planned (on the CPU: the plan reads no matrix), and on the GPU the edges of the copies, the queue's one
buffer shared by several commands under flushes, and a stream under capture, which gets no copies."""
import random
import time
from ctypes import byref, c_int32, c_uint64

import numpy as np
import pytest

TWO_BUFFERS, FOUR_STAGES, ANY_SHAPE = 0, 1, 2
EXACT, EDGES = 0, 1
COPIED_PER_GROUP = 256 * 4 * 8      # elements that a work-group copies


def plans_of(xs, a, b, c, M, N, K):
    """(launches as they lie, launches on copies, work-groups that copy A, and B)"""
    out = (c_int32 * 10)()
    parts = lambda: [tuple(out[i:i + 4]) for i in (0, 4) if out[i] != 0]
    xs.check(xs.halhip().HipGemmBf16PlanOf(a, b, c, M, N, K, out))
    in_place = parts()
    xs.check(xs.halhip().HipGemmBf16CopyPlanOf(a, b, c, M, N, K, out))
    return in_place, parts(), out[8], out[9]


def test_what_is_copied(xs):
    rng = random.Random(5)
    copied = 0
    for _ in range(8000):
        M, N, K = (int(2 ** rng.uniform(0, 14)) for _ in range(3))
        if rng.random() < 0.3:
            N = max(8, N // 8 * 8)
        if rng.random() < 0.3:
            K = max(8, K // 8 * 8)
        a, b, c = ((1 << 20) + rng.choice([0, 0, 0, 2]) for _ in range(3))
        in_place, parts, groups_a, groups_b = plans_of(xs, a, b, c, M, N, K)
        case = (M, N, K, a, b, c, in_place, parts, groups_a, groups_b)
        off_a, off_b = a % 16 != 0 or K % 8 != 0, b % 16 != 0 or N % 8 != 0
        if not parts:
            assert groups_a == groups_b == 0, case
            continue
        copied += 1
        assert in_place[0][2] != ANY_SHAPE, case
        assert (groups_a > 0, groups_b > 0) == (off_a, off_b) and (off_a or off_b), case
        for groups, rows, cols in ((groups_a, M, K), (groups_b, K, N)):
            if groups:
                assert groups == -(-rows * (-(-cols // 64) * 64) // COPIED_PER_GROUP), case
        assert sum(rows for rows, *_ in parts) == M, case
        tiles, heights = groups_a + groups_b, (c_int32 * 4)()
        xs.check(xs.halhip().HipGemmBf16TileRowsOf(a, b, c, M, N, K, heights))
        for (rows, edge, kernel, fit), height in zip(parts, heights[2:]):
            tiles += -(-rows // height) * -(-N // edge)
            whole = c % 16 == 0 and N % edge == 0 and rows % height == 0 and K % 64 == 0
            assert fit == (EXACT if whole else EDGES), case
        assert tiles <= 1 << 18, case
    assert copied > 300


def test_what_is_not_copied(xs, monkeypatch):
    at = 1 << 20
    assert plans_of(xs, at, at, at, 4001, 4003, 2048)[1] != []
    assert plans_of(xs, at, at, at + 2, 4096, 4096, 2048)[1] == []          # only C is off: nothing to copy
    assert plans_of(xs, at, at, at + 2, 4096, 4096, 2048)[0] == [(4096, 256, TWO_BUFFERS, EDGES)]
    assert plans_of(xs, at, at, at, 20001, 20003, 20001)[1] == []           # copies of 1.6 GB
    assert plans_of(xs, at, at, at, 300, 301, 303)[1] == []                 # copying takes longer than it saves
    monkeypatch.setenv("XSCHED_HIP_GEMM_TILE", "128")
    assert plans_of(xs, at, at, at, 4001, 4003, 2048)[1] == []


def test_thin_products_of_large_matrices_are_not_copied(xs):
    """Copies beyond the last-level cache cost two passes over memory, which a thin product does not win back."""
    at = 1 << 20
    for sizes in ((8191, 512, 8191), (512, 16383, 8191), (500, 12287, 8191), (16383, 300, 8191), (300, 16383, 8191)):
        assert plans_of(xs, at, at, at, *sizes)[1] == [], sizes
    for sizes in ((700, 8191, 8191), (8191, 1023, 8191), (8191, 2047, 8191), (1500, 8191, 4095), (8191, 8191, 8191)):
        assert plans_of(xs, at, at, at, *sizes)[1] != [], sizes


def test_copies_for_tiles_of_fewer_rows_only_where_they_gain(xs):
    """By the estimate alone all of these are quicker on copies."""
    at = 1 << 20
    for sizes in ((774, 6505, 1056), (1071, 3980, 1184), (1897, 3814, 1002), (897, 4134, 1120), (1440, 5114, 808), (1271, 4106, 1020)):
        assert plans_of(xs, at, at, at, *sizes)[1] == [], sizes
    for sizes in ((767, 5952, 1317), (1750, 4884, 336), (3207, 6144, 197), (610, 7424, 846), (817, 5008, 1301), (6754, 631, 2169), (640, 12001, 3801),
                  (730, 7489, 2278), (599, 7697, 2539)):
        assert plans_of(xs, at, at, at, *sizes)[1] == [(sizes[0], 256, TWO_BUFFERS, EDGES)], sizes


@pytest.mark.parametrize("M,N,K,copied", [
    (500, 499, 4095, False), (1500, 1499, 4095, True), (1500, 1499, 2047, False), (2000, 1999, 2047, False), (2000, 1999, 3001, False),
    (2000, 1999, 4095, True), (2500, 2501, 1001, False), (3000, 2999, 301, False), (3000, 2999, 101, False), (4000, 3999, 301, True),
    (1000, 999, 8001, False), (128, 8191, 8191, False)])
def test_the_way_of_the_products_that_were_timed_both_ways(xs, M, N, K, copied):
    assert (plans_of(xs, 1 << 20, 1 << 20, 1 << 20, M, N, K)[1] != []) == copied


def _ints(torch, gen, shape, offset):
    """Integers in [-2, 2] between NaNs, `offset` elements behind an aligned address."""
    rows, cols = shape
    flat = torch.full((rows * cols + offset + 64,), float("nan"), dtype=torch.bfloat16, device="cuda")
    flat[offset:offset + rows * cols] = torch.randint(-2, 3, (rows * cols,), device="cuda", generator=gen).to(torch.bfloat16)
    return flat[offset:offset + rows * cols].view(rows, cols)


# both, A alone, B alone; rows of one piece more or less than whole lines, the last piece of one and of
# seven elements, K of the last step 1 and 63; matrices off by an element; C alone off
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,offsets,copied", [
    (4000, 3999, 301, (0, 0, 0), "ab"), (3500, 3503, 1025, (0, 0, 0), "ab"), (3001, 3009, 1087, (1, 3, 5), "ab"),
    (3000, 3008, 1001, (0, 0, 0), "a"), (3000, 3001, 1000, (0, 0, 0), "b"), (4096, 4096, 1024, (1, 0, 0), "a"),
    (4096, 4096, 1024, (0, 7, 1), "b"), (4100, 4104, 1024, (0, 0, 1), "")])
@pytest.mark.parametrize("level,guard", [(1, 0), (2, 1)])
def test_gemm_on_copies(xs, gpu, M, N, K, offsets, copied, level, guard):
    """(K x 4 < 2^24: float32 sums are exact in any order.)"""
    from test_gpu_kernels import Queue, gemm_cmd
    torch = gpu
    print(f"case gemm-copies M={M} N={N} K={K} offsets={offsets} level={level} guard={guard}", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + K)
    a, b = _ints(torch, gen, (M, K), offsets[0]), _ints(torch, gen, (K, N), offsets[1])
    c_flat = torch.full((M * N + offsets[2] + 64,), 0.5, dtype=torch.bfloat16, device="cuda")
    c = c_flat[offsets[2]:offsets[2] + M * N].view(M, N)
    torch.cuda.synchronize()
    _, parts, groups_a, groups_b = plans_of(xs, a.data_ptr(), b.data_ptr(), c.data_ptr(), M, N, K)
    assert ("a" if groups_a else "") + ("b" if groups_b else "") == copied and bool(parts) == bool(copied)
    q = Queue(xs, torch, level)
    q.submit(gemm_cmd(xs, a, b, c, M, N, K, guard))
    q.wait()
    q.close()
    assert torch.equal(c, (a.float() @ b.float()).to(torch.bfloat16))
    assert bool((c_flat[:offsets[2]] == 0.5).all()) and bool((c_flat[offsets[2] + M * N:] == 0.5).all())


@pytest.mark.gpu
def test_copied_matrices_are_summed_in_the_same_order(xs, gpu, monkeypatch):
    """Normally distributed inputs: the same bits as through registers."""
    from test_gpu_kernels import Queue, gemm_cmd
    torch = gpu
    M, N, K = 3001, 2999, 1001
    print(f"case gemm-copies-order M={M} N={N} K={K}", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(1)
    a, b = (torch.randn(s, device="cuda", generator=gen).to(torch.bfloat16) for s in ((M, K), (K, N)))
    got, want = (torch.zeros(M, N, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    torch.cuda.synchronize()
    assert plans_of(xs, a.data_ptr(), b.data_ptr(), got.data_ptr(), M, N, K)[1] != []
    q = Queue(xs, torch, 2)
    q.submit(gemm_cmd(xs, a, b, got, M, N, K, 1))
    monkeypatch.setenv("XSCHED_HIP_GEMM_TILE", "128")
    q.submit(gemm_cmd(xs, a, b, want, M, N, K, 1))
    q.wait()
    q.close()
    assert torch.equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("forced", ["", "128"])
def test_commands_that_share_the_buffer_flushed_and_replayed(xs, gpu, monkeypatch, forced):
    """Three products in flight, of different matrices and sizes, whose copies go to the same buffer one
    after the other: suspended at a random moment and resumed, until one has been flushed in
    the middle three times. (Forced to 128 x 128 tiles: the same through registers, without copies. Other work keeps
    compute units busy: without it all tiles of a product start at once, and 250 to 450 of the 600 rounds were needed.)"""
    from test_gemm_split import Busy, Moment
    from test_gpu_kernels import Queue, gemm_cmd
    from test_gpu_preempt import hip_stats
    torch = gpu
    if forced:
        monkeypatch.setenv("XSCHED_HIP_GEMM_TILE", forced)
    print(f"case gemm-copies-flush forced={forced}", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(3)
    products = []
    for M, N, K in ((3001, 3003, 1001), (4001, 4003, 2047), (2999, 3500, 1500)):
        a, b = _ints(torch, gen, (M, K), 0), _ints(torch, gen, (K, N), 1)
        c = torch.zeros(M, N, dtype=torch.bfloat16, device="cuda")
        assert (plans_of(xs, a.data_ptr(), b.data_ptr(), c.data_ptr(), M, N, K)[1] == []) == bool(forced)
        products.append((a, b, c, (a.float() @ b.float()).to(torch.bfloat16)))
    q, p, busy = Queue(xs, torch, 2), xs.preempt(), Busy(torch)

    def submit():
        busy.begin()
        for a, b, c, _ in products:
            q.submit(gemm_cmd(xs, a, b, c, a.shape[0], b.shape[1], a.shape[1], 1))
    torch.cuda.synchronize()
    for _ in range(3):
        began = time.perf_counter()
        submit()
        q.wait()
        span = time.perf_counter() - began
        torch.cuda.synchronize()
    flushed, rounds, moment = 0, 0, Moment(3, span)
    while flushed < 3 and rounds < 3000:
        rounds += 1
        for _, _, c, _ in products:
            c.fill_(float("nan"))
        torch.cuda.synchronize()
        submit()
        moment.wait()
        xs.check(p.XQueueSuspend(q.xq, xs.kQueueSuspendFlagSyncHwQueue))
        missing = [torch.isnan(c) for _, _, c, _ in products]
        moment.met(missing[0], missing[-1])
        some = any(bool(m.any()) and not bool(m.all()) for m in missing)
        xs.check(p.XQueueResume(q.xq, xs.kQueueResumeFlagNone))
        q.wait()
        for i, (_, _, c, want) in enumerate(products):
            assert torch.equal(c, want), f"product {i}, round {rounds}, flushed in the middle: {some}"
        flushed += some
    st = hip_stats(xs, q.hwq)
    torch.cuda.synchronize()
    q.close()
    print("stats", st, "rounds", rounds, "flushed in the middle", flushed, flush=True)
    assert flushed == 3 and st[1] >= 3


@pytest.mark.gpu
def test_a_captured_product_uses_no_buffer_of_the_queue(xs, gpu):
    """A graph outlives the command and its queue: under capture the matrices are read where they lie.
    Replayed three times after the queue is gone, with other work in between."""
    torch = gpu
    M, N, K = 3001, 2999, 1001
    print(f"case gemm-copies-capture M={M} N={N} K={K}", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(2)
    a, b = _ints(torch, gen, (M, K), 0), _ints(torch, gen, (K, N), 0)
    c = torch.zeros(M, N, dtype=torch.bfloat16, device="cuda")
    want = (a.float() @ b.float()).to(torch.bfloat16)
    p, h, stream = xs.preempt(), xs.halhip(), torch.cuda.Stream()
    hwq = xs.hip_queue_create(stream.cuda_stream)

    def launch():
        cmd = c_uint64()
        xs.check(h.HipGemmBf16CommandCreate(byref(cmd), a.data_ptr(), b.data_ptr(), c.data_ptr(), M, N, K, 0))
        xs.check(p.HwQueueLaunch(hwq, cmd.value))
    assert plans_of(xs, a.data_ptr(), b.data_ptr(), c.data_ptr(), M, N, K)[1] != []
    torch.cuda.synchronize()
    launch()                            # eagerly first: on copies
    stream.synchronize()
    assert torch.equal(c, want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        launch()
    torch.cuda.synchronize()
    xs.check(p.HwQueueDestroy(hwq))
    other = torch.zeros(1 << 26, device="cuda")   # may lie where the queue's buffer was
    for replay in range(3):
        c.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(c, want), f"replay {replay}"
        other.add_(1.0)
        torch.cuda.synchronize()
    assert bool((other == 3.0).all())
