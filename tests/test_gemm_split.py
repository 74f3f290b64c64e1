"""Products whose K is divided among work-groups: when that is planned (on the CPU: the plan reads no
matrix), and on the GPU the edges of parts and tiles, the sums' error, flushes between the parts of a tile, commands one
behind the other on the same ticket words, and a stream under capture, where nothing is divided."""
import random
import time
from ctypes import byref, c_int32, c_uint64

import pytest


def splits_of(xs, a, b, c, M, N, K):
    out = (c_int32 * 2)()
    xs.check(xs.halhip().HipGemmBf16SplitsOf(a, b, c, M, N, K, out))
    return out[0], out[1]


def test_what_is_split(xs, monkeypatch):
    rng = random.Random(11)
    at, split, whole = 1 << 20, 0, 0
    for _ in range(4000):
        M, N, K = (int(2 ** rng.uniform(0, 14)) for _ in range(3))
        if rng.random() < 0.5:
            N, K = max(8, N // 8 * 8), max(64, K // 64 * 64)
        plan = (c_int32 * 8)()
        xs.check(xs.halhip().HipGemmBf16PlanOf(at, at, at, M, N, K, plan))
        parts, on_copies = splits_of(xs, at, at, at, M, N, K)
        case = (M, N, K, list(plan), parts, on_copies)
        if parts == 1:
            whole += 1
            continue
        split += 1
        rows, tile, kernel, _ = plan[:4]
        tiles = -(-M // tile) * -(-N // tile)
        assert plan[4] == 0 and rows == M and kernel == 1 and tile in (64, 128), case
        assert tiles * parts <= 256 and K > 1024 and parts <= -(-K // 64 // 8), case
    assert split > 200 and whole > 2000
    assert splits_of(xs, at, at, at, 256, 256, 8192)[0] > 4
    assert splits_of(xs, at, at, at, 256, 256, 1024) == (1, 0)
    assert splits_of(xs, at, at, at, 1024, 1024, 1024) == (1, 0)          # a tile for every compute unit
    assert splits_of(xs, at, at, at, 4096, 4096, 8192) == (1, 0)
    monkeypatch.setenv("XSCHED_HIP_GEMM_TILE", "64")
    assert splits_of(xs, at, at, at, 256, 256, 8192) == (1, 0)


def _ints(torch, gen, shape, offset):
    """Integers in [-2, 2] between NaNs, `offset` elements behind an aligned address."""
    rows, cols = shape
    flat = torch.full((rows * cols + offset + 64,), float("nan"), dtype=torch.bfloat16, device="cuda")
    flat[offset:offset + rows * cols] = torch.randint(-2, 3, (rows * cols,), device="cuda", generator=gen).to(torch.bfloat16)
    return flat[offset:offset + rows * cols].view(rows, cols)


# whole tiles; ragged rows, columns and last step on 16-byte boundaries; any sizes and offsets through registers, the last
# step of 1 and of 63 values; a last part shorter than the others; tiles of 128; one tile; copies of A, of B
SHAPES = [(128, 128, 8192, 0), (64, 64, 2048, 0), (256, 320, 4096, 0), (130, 200, 4104, 0), (65, 72, 2040, 0), (300, 301, 3009, 0),
          (63, 65, 4095, 1), (100, 9, 2111, 3), (1024, 1024, 8192, 0), (1000, 1016, 8008, 0), (700, 701, 8001, 1), (1, 8, 8192, 0)]


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,offset", SHAPES)
@pytest.mark.parametrize("level,guard", [(1, 0), (2, 1)])
def test_gemm_split(xs, gpu, M, N, K, offset, level, guard):
    """Twice: the second command finds the tickets of the first. (K x 4 < 2^24: float32 sums are exact in any
    order.)"""
    from test_gpu_kernels import Queue, gemm_cmd
    torch = gpu
    print(f"case gemm-split M={M} N={N} K={K} offset={offset} level={level} guard={guard}", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + K)
    a, b = _ints(torch, gen, (M, K), offset), _ints(torch, gen, (K, N), offset)
    flat = [torch.full((M * N + offset + 64,), 0.5, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    cs = [f[offset:offset + M * N].view(M, N) for f in flat]
    torch.cuda.synchronize()
    assert max(splits_of(xs, a.data_ptr(), b.data_ptr(), cs[0].data_ptr(), M, N, K)) > 1
    q = Queue(xs, torch, level)
    for c in cs:
        q.submit(gemm_cmd(xs, a, b, c, M, N, K, guard))
    q.wait()
    q.close()
    want = (a.double() @ b.double()).to(torch.bfloat16)
    for f, c in zip(flat, cs):
        assert torch.equal(c, want)
        assert bool((f[:offset] == 0.5).all()) and bool((f[offset + M * N:] == 0.5).all())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(128, 128, 8192), (300, 301, 3009), (1024, 1024, 8192)])
def test_split_sums_are_as_good_as_whole_ones_and_always_the_same(xs, gpu, monkeypatch, M, N, K):
    """Normally distributed inputs: no further from the product in 64 bits than in one go (the rounding to bf16
    is nearly all of either, a hundredth is left for it), and whoever draws the last ticket, the same bits."""
    from test_gpu_kernels import Queue, gemm_cmd
    torch = gpu
    print(f"case gemm-split-error M={M} N={N} K={K}", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(K)
    a, b = (torch.randn(s, device="cuda", generator=gen).to(torch.bfloat16) for s in ((M, K), (K, N)))
    cs = [torch.zeros(M, N, dtype=torch.bfloat16, device="cuda") for _ in range(21)]
    torch.cuda.synchronize()
    q = Queue(xs, torch, 2)
    for c in cs[:20]:
        q.submit(gemm_cmd(xs, a, b, c, M, N, K, 1))
    monkeypatch.setenv("XSCHED_HIP_GEMM_TILE", "64")
    q.submit(gemm_cmd(xs, a, b, cs[20], M, N, K, 1))
    q.wait()
    q.close()
    want = a.double() @ b.double()
    error = [float((c.double() - want).norm() / want.norm()) for c in (cs[0], cs[20])]
    print("error split", error[0], "whole", error[1], flush=True)
    assert error[0] <= 1.01 * error[1]
    assert all(torch.equal(c, cs[0]) for c in cs[1:20])


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [((512, 1024, 8192), (1024, 1024, 8192)), ((700, 701, 8001), (200, 300, 8192))])
def test_split_commands_flushed_and_replayed(xs, gpu, sizes):
    """Commands of two shapes in turn, whose parts and tickets lie in the same places: suspended at a random moment and
    resumed, until commands have been flushed and replayed forty times."""
    from test_gpu_kernels import Queue, gemm_cmd
    from test_gpu_preempt import hip_stats
    torch = gpu
    print(f"case gemm-split-flush sizes={sizes}", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)
    products = []
    for M, N, K in sizes * 3:
        a, b = _ints(torch, gen, (M, K), 0), _ints(torch, gen, (K, N), 0)
        c = torch.zeros(M, N, dtype=torch.bfloat16, device="cuda")
        assert max(splits_of(xs, a.data_ptr(), b.data_ptr(), c.data_ptr(), M, N, K)) > 1
        products.append((a, b, c, (a.double() @ b.double()).to(torch.bfloat16)))
    q, p, rnd = Queue(xs, torch, 2), xs.preempt(), random.Random(7)

    def submit():
        for a, b, c, _ in products:
            q.submit(gemm_cmd(xs, a, b, c, a.shape[0], b.shape[1], a.shape[1], 1))
    torch.cuda.synchronize()
    submit()
    q.wait()
    began = time.perf_counter()
    submit()
    q.wait()
    span = time.perf_counter() - began
    rounds = 0
    while hip_stats(xs, q.hwq)[1] < 40 and rounds < 600:
        rounds += 1
        for _, _, c, _ in products:
            c.fill_(float("nan"))
        torch.cuda.synchronize()
        submit()
        until = time.perf_counter() + rnd.uniform(0.0, 1.2 * span)
        while time.perf_counter() < until:
            pass
        xs.check(p.XQueueSuspend(q.xq, xs.kQueueSuspendFlagSyncHwQueue))
        xs.check(p.XQueueResume(q.xq, xs.kQueueResumeFlagNone))
        q.wait()
        for i, (_, _, c, want) in enumerate(products):
            assert torch.equal(c, want), f"product {i}, round {rounds}"
    st = hip_stats(xs, q.hwq)
    q.close()
    print("stats", st, "rounds", rounds, flush=True)
    assert st[1] >= 40


@pytest.mark.gpu
def test_a_captured_product_is_not_split(xs, gpu):
    """A graph outlives the command and its queue: what it holds uses no memory of theirs. Replayed three times after the
    queue is gone, with other work in between."""
    torch = gpu
    M, N, K = 256, 256, 8192
    print(f"case gemm-split-capture M={M} N={N} K={K}", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(2)
    a, b = _ints(torch, gen, (M, K), 0), _ints(torch, gen, (K, N), 0)
    c = torch.zeros(M, N, dtype=torch.bfloat16, device="cuda")
    want = (a.double() @ b.double()).to(torch.bfloat16)
    p, h, stream = xs.preempt(), xs.halhip(), torch.cuda.Stream()
    hwq = xs.hip_queue_create(stream.cuda_stream)

    def launch():
        cmd = c_uint64()
        xs.check(h.HipGemmBf16CommandCreate(byref(cmd), a.data_ptr(), b.data_ptr(), c.data_ptr(), M, N, K, 0))
        xs.check(p.HwQueueLaunch(hwq, cmd.value))
    assert splits_of(xs, a.data_ptr(), b.data_ptr(), c.data_ptr(), M, N, K)[0] > 1
    torch.cuda.synchronize()
    launch()                            # eagerly first: split
    stream.synchronize()
    assert torch.equal(c, want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        launch()
    torch.cuda.synchronize()
    xs.check(p.HwQueueDestroy(hwq))
    other = torch.zeros(1 << 24, device="cuda")   # may lie where the queue's buffer was
    for replay in range(3):
        c.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(c, want), f"replay {replay}"
        other.add_(1.0)
        torch.cuda.synchronize()
    assert bool((other == 3.0).all())
