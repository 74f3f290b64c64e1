"""Large tiles of 192 and 128 rows: the rule that takes them, on the CPU, and on the GPU their
edges and the lengths of their pipeline."""
import random
from ctypes import byref, c_int32, c_uint64

import numpy as np
import pytest

import oracle

ADDRESS = 1 << 20


def tile_rows_of(xs, a, b, c, M, N, K):
    out = (c_int32 * 4)()
    xs.check(xs.halhip().HipGemmBf16TileRowsOf(a, b, c, M, N, K, out))
    return list(out)


@pytest.mark.parametrize("M,N,K,rows", [
    (4096, 4096, 4096, 256), (8192, 8192, 8192, 256), (3072, 3072, 3072, 192), (3456, 3456, 512, 192), (7451, 2632, 1232, 192),
    (5801, 760, 3344, 128), (805, 7704, 104, 128), (1500, 5240, 592, 128), (2048, 2048, 2048, 128), (1024, 1024, 1024, 64),
    # behind a whole round, where two launches are the other way
    (4608, 4608, 4608, 192), (4994, 6840, 456, 192), (3488, 5808, 464, 192), (7680, 3072, 3840, 192), (2624, 7296, 6400, 192), (5124, 4096, 2048, 192)])
def test_the_rows_that_measured_quickest_are_taken(xs, M, N, K, rows):
    assert tile_rows_of(xs, ADDRESS, ADDRESS, ADDRESS, M, N, K)[:2] == [rows, 0]


@pytest.mark.parametrize("M,N,K", [(4996, 4096, 2048), (3840, 4608, 2048), (6896, 2448, 2816), (3199, 5120, 6848), (7024, 2792, 4160)])
def test_two_launches_that_measured_quickest_are_kept(xs, M, N, K):
    first, second = tile_rows_of(xs, ADDRESS, ADDRESS, ADDRESS, M, N, K)[:2]
    assert first == 256 and second != 0


def counted_tiles(M, N, K):
    """By which a product of matrices on 16-byte boundaries is accepted, up to 2^18."""
    tiles = lambda rows, edge: -(-rows // edge) * -(-N // edge)
    whole = M // 128 * 128
    if whole == 0 or N % 128 != 0 or K % 64 != 0:
        return tiles(M, 64)
    return tiles(whole, 256 if whole % 256 == 0 and N % 256 == 0 else 128) + tiles(M - whole, 64)


def test_tiles_of_fewer_rows_stay_within_what_the_progress_map_holds(xs):
    """And no product is refused for them."""
    rng = random.Random(3)
    seen, too_many = set(), 0
    for _ in range(6000):
        M, N, K = int(2 ** rng.uniform(6, 24)), int(2 ** rng.uniform(6, 14)) // 8 * 8, 64 * rng.randint(1, 64)
        if rng.random() < 0.3:      # about the limit, a multiple of the tiles
            N = max(256, N // 256 * 256)
            M = int((1 << 18) / (N // 256) * rng.uniform(0.4, 1.02)) * 256
        plan, cmd = (c_int32 * 8)(), c_uint64()
        xs.check(xs.halhip().HipGemmBf16PlanOf(ADDRESS, ADDRESS, ADDRESS, M, N, K, plan))
        rows = tile_rows_of(xs, ADDRESS, ADDRESS, ADDRESS, M, N, K)
        case = (M, N, K, list(plan), rows)
        taken = xs.halhip().HipGemmBf16CommandCreate(byref(cmd), ADDRESS, ADDRESS, ADDRESS, M, N, K, 1) == xs.kXSchedSuccess
        assert taken == (counted_tiles(M, N, K) <= 1 << 18), case
        if not taken:
            continue
        xs.check(xs.preempt().HwCommandDestroy(cmd.value))
        assert sum(-(-plan[4 * i] // rows[i]) * -(-N // plan[4 * i + 1]) for i in range(2) if rows[i]) <= 1 << 18, case
        seen.update((rows[i], plan[4 * i + 1]) for i in range(2) if rows[i])
        too_many += -(-M // 192) * -(-N // 256) > 1 << 18
    assert {(256, 256), (192, 256), (128, 256), (128, 128), (64, 64)} <= seen
    assert too_many > 100       # 192 rows would not fit there, 256 do


@pytest.mark.gpu
@pytest.mark.parametrize("level,guard", [(1, 0), (2, 1)])
@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5, 6, 7, 8, 9, 13, 18])
@pytest.mark.parametrize("fit", ["exact", "edges", "one row"])
@pytest.mark.parametrize("rows", [192, 128])
def test_pipeline_lengths_and_edges(xs, gpu, monkeypatch, rows, fit, steps, level, guard):
    """Integers in [-4, 4] (at most 18 x 64 x 16 < 2^24): every sum is exact. The matrices lie between NaNs, C
    between values that must come back untouched."""
    from test_gpu_kernels import Queue
    torch, pad = gpu, 8
    monkeypatch.setenv("XSCHED_HIP_GEMM_TILE", "256")
    monkeypatch.setenv("XSCHED_HIP_GEMM_TILE_ROWS", str(rows))
    M, N, K = {"exact": (2 * rows, 512, 64 * steps), "edges": (2 * rows - 1, 264, 64 * steps - 8 * (1 + (steps - 1) % 7)),
               "one row": (rows + 1, 248, 64 * steps - 56)}[fit]
    print(f"case gemm-tile-rows rows={rows} M={M} N={N} K={K} level={level} guard={guard}", flush=True)
    rng = np.random.default_rng(100 * steps + rows)
    nan = 0x7FC0

    def between_nans(bits):
        return np.concatenate([np.full(pad, nan, np.uint16), bits.ravel(), np.full(64, nan, np.uint16)])
    a_bits = oracle.f32_to_bf16_bits(rng.integers(-4, 5, (M, K)).astype(np.float32))
    b_bits = oracle.f32_to_bf16_bits(rng.integers(-4, 5, (K, N)).astype(np.float32))
    a = torch.from_numpy(between_nans(a_bits).view(np.int16)).cuda()
    b = torch.from_numpy(between_nans(b_bits).view(np.int16)).cuda()
    c = torch.full((pad + M * N + 64,), 0x1234, dtype=torch.int16, device="cuda")
    at = a.data_ptr() + 2 * pad, b.data_ptr() + 2 * pad, c.data_ptr() + 2 * pad
    assert tile_rows_of(xs, *at, M, N, K)[0] == rows
    q, cmd = Queue(xs, torch, level), c_uint64()
    xs.check(xs.halhip().HipGemmBf16CommandCreate(byref(cmd), *at, M, N, K, guard))
    q.submit(cmd.value)
    q.wait()
    got = c.cpu().numpy().view(np.uint16)
    q.close()
    want = oracle.gemm_bf16(a_bits.ravel(), b_bits.ravel(), M, N, K)
    assert np.array_equal(got[pad:pad + M * N].reshape(M, N), want.reshape(M, N))
    assert np.all(got[:pad] == 0x1234) and np.all(got[pad + M * N:] == 0x1234)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,sizes", [(192, (3072, 3080, 2048)), (128, (2000, 2048, 2056))])
def test_the_same_bits_as_square_tiles_flushed_and_replayed(xs, gpu, monkeypatch, rows, sizes):
    """Normally distributed inputs: every tile adds an element's products in the same order, also where a product is suspended
    at any moment and resumed."""
    import threading

    from test_gpu_kernels import Queue, gemm_cmd
    from test_gpu_preempt import churn, hip_stats
    torch = gpu
    M, N, K = sizes
    print(f"case gemm-tile-rows-replayed rows={rows} {sizes}", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(2)
    a, b = (torch.randn(*s, device="cuda", generator=gen).to(torch.bfloat16) for s in ((M, K), (K, N)))
    monkeypatch.setenv("XSCHED_HIP_GEMM_TILE", "128")
    want = torch.zeros(M, N, dtype=torch.bfloat16, device="cuda")
    torch.cuda.synchronize()
    q = Queue(xs, torch, 1)
    q.submit(gemm_cmd(xs, a, b, want, M, N, K, 0))
    q.wait()
    q.close()
    monkeypatch.setenv("XSCHED_HIP_GEMM_TILE", "256")
    monkeypatch.setenv("XSCHED_HIP_GEMM_TILE_ROWS", str(rows))
    outs = [torch.full_like(want, float("nan")) for _ in range(40)]
    torch.cuda.synchronize()
    q, stop = Queue(xs, torch, 2, threshold=4, batch=2), threading.Event()
    t = threading.Thread(target=churn, args=(xs, q, stop, 3))
    t.start()
    for c in outs:
        q.submit(gemm_cmd(xs, a, b, c, M, N, K, 1))
    q.wait()
    stop.set()
    t.join()
    st = hip_stats(xs, q.hwq)
    q.close()
    print("stats", st, flush=True)
    assert st[2] > 0
    assert [i for i, c in enumerate(outs) if not torch.equal(c, want)] == []
