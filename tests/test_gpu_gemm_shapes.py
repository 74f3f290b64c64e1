"""GPU parity of the GEMM's tile kernels at the sizes where they change their ways: the number
of K steps around the length of their pipelines and of their polls of the preempt word, the last
step full and not, edges of tiles, and rows that start on 16-byte boundaries or do not."""
import time
from ctypes import byref, c_int32, c_uint64

import numpy as np
import pytest

import oracle
from test_gemm_split import Busy, Moment
from test_gpu_kernels import Queue, gemm_cmd
from test_gpu_preempt import hip_stats

pytestmark = pytest.mark.gpu

NAN = 0x7FC0
TWO_BUFFERS, FOUR_STAGES, ANY_SHAPE = 0, 1, 2      # kernels of a plan


def plan_of(xs, a, b, c, M, N, K):
    """[(rows, tile, kernel, fit)] of the one or two launches of a GEMM."""
    out = (c_int32 * 8)()
    xs.check(xs.halhip().HipGemmBf16PlanOf(a.data_ptr(), b.data_ptr(), c.data_ptr(), M, N, K, out))
    return [tuple(out[i:i + 4]) for i in (0, 4) if out[i] != 0]


def _shape(fit, tile, steps):
    if fit == "exact":
        return tile, 2 * tile, 64 * steps
    if fit == "edges":      # one row and eight columns in the second tile; 8 to 56 values in the last step
        return tile + 1, tile + 8, 64 * steps - 8 * (1 + (steps - 1) % 7)
    return tile + 3, tile + 1, 64 * steps - (2 * steps + 1) % 64   # odd sizes


@pytest.mark.parametrize("level,guard", [(1, 0), (2, 1)])
@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5, 6, 7, 9, 10, 13, 14, 18])
@pytest.mark.parametrize("tile,fit", [(t, f) for t in (64, 128) for f in ("exact", "edges", "unaligned")] + [(256, "exact"), (256, "edges")])
def test_gemm_pipeline_lengths_and_edges(xs, gpu, monkeypatch, tile, fit, steps, level, guard):
    """Integers in [-4, 4]: at most 18 x 64 x 16 < 2^24, so every sum is exact and the result is
    determined. The matrices lie between NaNs, which must not get into a sum, and C between
    values that must come back untouched."""
    torch = gpu
    monkeypatch.setenv("XSCHED_HIP_GEMM_TILE", str(tile))
    M, N, K = _shape(fit, tile, steps)
    pad = 3 if fit == "unaligned" else 8     # elements in front of each matrix
    print(f"case gemm-pipeline tile={tile} {fit} M={M} N={N} K={K} level={level} guard={guard}", flush=True)
    rng = np.random.default_rng(100 * steps + tile)

    def between_nans(bits):
        return np.concatenate([np.full(pad, NAN, np.uint16), bits.ravel(), np.full(64, NAN, np.uint16)])
    a_bits = oracle.f32_to_bf16_bits(rng.integers(-4, 5, (M, K)).astype(np.float32))
    b_bits = oracle.f32_to_bf16_bits(rng.integers(-4, 5, (K, N)).astype(np.float32))
    a = torch.from_numpy(between_nans(a_bits).view(np.int16)).cuda()
    b = torch.from_numpy(between_nans(b_bits).view(np.int16)).cuda()
    c = torch.full((pad + M * N + 64,), 0x1234, dtype=torch.int16, device="cuda")
    q = Queue(xs, torch, level)
    cmd = c_uint64()
    xs.check(xs.halhip().HipGemmBf16CommandCreate(byref(cmd), a.data_ptr() + 2 * pad, b.data_ptr() + 2 * pad,
                                                  c.data_ptr() + 2 * pad, M, N, K, guard))
    q.submit(cmd.value)
    q.wait()
    got = c.cpu().numpy().view(np.uint16)
    q.close()
    want = oracle.gemm_bf16(a_bits.ravel(), b_bits.ravel(), M, N, K)
    assert np.array_equal(got[pad:pad + M * N].reshape(M, N), want.reshape(M, N))
    assert np.all(got[:pad] == 0x1234) and np.all(got[pad + M * N:] == 0x1234)


@pytest.mark.parametrize("M,N,K", [(4100, 4096, 512), (4096 + 257, 4096, 520), (8450, 2056, 448), (2100, 8192, 456)])
@pytest.mark.parametrize("flush", [False, True])
def test_gemm_in_two_launches(xs, gpu, M, N, K, flush):
    """Rows that fill whole rounds of large tiles in one launch, the rest on smaller tiles in
    another, one command: with the queue suspended and resumed at once behind each, too (flushed in the
    middle: test_gemm_flushed_and_replayed). Integers
    in [-4, 4] (K x 16 < 2^24): float32 sums are exact in any order."""
    torch = gpu
    print(f"case gemm-two-launches M={M} N={N} K={K} flush={flush}", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + K)
    a, b = (torch.randint(-4, 5, s, device="cuda", generator=gen).to(torch.bfloat16) for s in ((M, K), (K, N)))
    cs = [torch.full((M + 2, N), 0.5, dtype=torch.bfloat16, device="cuda") for _ in range(6 if flush else 1)]
    torch.cuda.synchronize()
    assert len(plan_of(xs, a, b, cs[0], M, N, K)) == 2
    q, p = Queue(xs, torch, 2), xs.preempt()
    for c in cs:
        cmd = c_uint64()
        xs.check(xs.halhip().HipGemmBf16CommandCreate(byref(cmd), a.data_ptr(), b.data_ptr(), c.data_ptr(), M, N, K, 1))
        q.submit(cmd.value)
        if flush:
            xs.check(p.XQueueSuspend(q.xq, xs.kQueueSuspendFlagSyncHwQueue))
            xs.check(p.XQueueResume(q.xq, xs.kQueueResumeFlagNone))
    q.wait()
    q.close()
    want = (a.float() @ b.float()).to(torch.bfloat16)
    for c in cs:
        assert torch.equal(c[:M], want)
        assert bool((c[M:] == 0.5).all()), "wrote behind the last row"


# 257 to 512 tiles of 128 x 128, and short K: K of one step, two, and around the polls of the preempt word
@pytest.mark.parametrize("M,N,K", [(2048, 2944, 64), (2048, 2944, 128), (1920, 2944, 192), (3968, 4224, 64), (1920, 2944, 320),
                                   (1920, 2944, 384), (2560, 2560, 704)])
@pytest.mark.parametrize("level,guard", [(1, 0), (2, 1)])
def test_gemm_two_work_groups_to_a_compute_unit(xs, gpu, monkeypatch, M, N, K, level, guard):
    """The kernel with two LDS buffers on 128 x 128 tiles. Its sums run in the order of the kernel
    with four stages on the same tiles: the same bits for normally distributed inputs."""
    torch = gpu
    print(f"case gemm-two-per-unit M={M} N={N} K={K} level={level} guard={guard}", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + K)
    a, b = (torch.randn(s, device="cuda", generator=gen).to(torch.bfloat16) for s in ((M, K), (K, N)))
    c = torch.full((M + 2, N), 0.5, dtype=torch.bfloat16, device="cuda")
    want = torch.zeros(M, N, dtype=torch.bfloat16, device="cuda")
    torch.cuda.synchronize()
    assert plan_of(xs, a, b, c, M, N, K) == [(M, 128, TWO_BUFFERS, 0)]
    q = Queue(xs, torch, level)
    q.submit(gemm_cmd(xs, a, b, c, M, N, K, guard))
    monkeypatch.setenv("XSCHED_HIP_GEMM_TILE", "128")
    assert plan_of(xs, a, b, want, M, N, K) == [(M, 128, FOUR_STAGES, 0)]
    q.submit(gemm_cmd(xs, a, b, want, M, N, K, guard))
    q.wait()
    q.close()
    # 2^-8 for the result's rounding to bf16, the rest for sums in another order
    torch.testing.assert_close(c[:M].float(), a.float() @ b.float(), rtol=2 ** -7, atol=2 ** -8 * K ** 0.5)
    assert torch.equal(c[:M], want)
    assert bool((c[M:] == 0.5).all()), "wrote behind the last row"


@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (8, 9, 1), (64, 72, 16), (65, 129, 31), (130, 72, 32), (63, 200, 8), (129, 65, 17), (300, 1, 257), (33, 7, 64)])
@pytest.mark.parametrize("pad", [8, 3])
@pytest.mark.parametrize("level,guard", [(1, 0), (2, 1)])
def test_gemm_any_shape_kernel(xs, gpu, M, N, K, pad, level, guard):
    """Short K and fewer than eight columns, with rows on 16-byte boundaries and off them, between
    NaNs that must not get into a sum. Integers: the result is determined."""
    torch = gpu
    print(f"case gemm-any-kernel M={M} N={N} K={K} pad={pad} level={level} guard={guard}", flush=True)
    rng = np.random.default_rng(K + 7)
    a_bits, b_bits = (oracle.f32_to_bf16_bits(rng.integers(-4, 5, s).astype(np.float32)) for s in ((M, K), (K, N)))

    def between_nans(bits):
        return torch.from_numpy(np.concatenate([np.full(pad, NAN, np.uint16), bits.ravel(), np.full(64, NAN, np.uint16)]).view(np.int16)).cuda()
    a, b = between_nans(a_bits), between_nans(b_bits)
    c = torch.full((pad + M * N + 64,), 0x1234, dtype=torch.int16, device="cuda")
    assert plan_of(xs, a[pad:], b[pad:], c[pad:], M, N, K) == [(M, 64, ANY_SHAPE, 2)]
    q = Queue(xs, torch, level)
    q.submit(gemm_cmd(xs, a[pad:], b[pad:], c[pad:], M, N, K, guard))
    q.wait()
    got = c.cpu().numpy().view(np.uint16)
    q.close()
    want = oracle.gemm_bf16(a_bits.ravel(), b_bits.ravel(), M, N, K)
    assert np.array_equal(got[pad:pad + M * N].reshape(M, N), want.reshape(M, N))
    assert np.all(got[:pad] == 0x1234) and np.all(got[pad + M * N:] == 0x1234)


@pytest.mark.parametrize("M,N,K,other", [(4097, 4099, 120, "128"), (4097, 4099, 120, "64"), (2000, 1999, 32, "64"), (300, 5, 1000, "wide"),
                                         (300, 5, 999, "wide"), (2000, 2000, 24, "256")])
def test_gemm_any_shape_kernel_adds_in_the_order_of_the_others(xs, gpu, monkeypatch, M, N, K, other):
    """Normally distributed inputs, where the order of the fp32 additions shows in the last bits: the
    same bits as on the tiles of another kernel, or, for few columns, as the same columns
    of a wider product."""
    torch = gpu
    print(f"case gemm-any-order M={M} N={N} K={K} {other}", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(K)
    cols = 64 if other == "wide" else N
    a, wide = (torch.randn(s, device="cuda", generator=gen).to(torch.bfloat16) for s in ((M, K), (K, cols)))
    b = wide[:, :N].contiguous()
    got, want = (torch.zeros(M, n, dtype=torch.bfloat16, device="cuda") for n in (N, cols))
    torch.cuda.synchronize()
    assert [p[2] for p in plan_of(xs, a, b, got, M, N, K)] == [ANY_SHAPE]
    q = Queue(xs, torch, 2)
    q.submit(gemm_cmd(xs, a, b, got, M, N, K, 1))
    if other != "wide":
        monkeypatch.setenv("XSCHED_HIP_GEMM_TILE", other)
    assert all(p[2] != ANY_SHAPE for p in plan_of(xs, a, wide, want, M, cols, K))
    q.submit(gemm_cmd(xs, a, wide, want, M, cols, K, 1))
    q.wait()
    q.close()
    assert torch.equal(got, want[:, :N])


@pytest.mark.parametrize("M,N,K,want_plan", [
    (1 << 18, 7, 512, [(64, ANY_SHAPE)]),                               # few columns
    (7001, 7003, 128, [(64, ANY_SHAPE)]),                               # short K
    (2560, 2560, 4096, [(128, TWO_BUFFERS)]),                           # two work-groups to a compute unit
    (4000, 4008, 4096, [(256, TWO_BUFFERS)]),                           # ragged large tiles
    (4001, 4003, 2048, [(128, FOUR_STAGES)]),                           # through registers
    # two launches (70.1 us, 74.9 on tiles of 192 rows; at 5124 rows, one launch on those, 84.0 and 75.5)
    (4868, 4096, 2048, [(256, TWO_BUFFERS), (128, FOUR_STAGES)])])
def test_gemm_flushed_and_replayed(xs, gpu, M, N, K, want_plan):
    """The queue is suspended at a random moment of a command until that has flushed it in the
    middle three times (C holds some tiles and not others; of two launches: all of the first one's and
    not all of the second's), then resumed each time: the replay does what is missing and nothing
    else. Other work keeps compute units busy: without it the 256 tiles of 4001 x 4003 x 2048 on copies all start at
    once, and 600 rounds met two such moments. Integers in [-2, 2] (K x 4 < 2^24): float32 sums are exact in any order."""
    torch = gpu
    print(f"case gemm-flush M={M} N={N} K={K}", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + K)
    a, b = (torch.randint(-2, 3, s, device="cuda", generator=gen).to(torch.bfloat16) for s in ((M, K), (K, N)))
    c = torch.zeros(M, N, dtype=torch.bfloat16, device="cuda")
    plan = plan_of(xs, a, b, c, M, N, K)
    assert [(p[1], p[2]) for p in plan] == want_plan, plan
    want = (a.float() @ b.float()).to(torch.bfloat16)
    q, p, busy = Queue(xs, torch, 2), xs.preempt(), Busy(torch)
    torch.cuda.synchronize()
    for _ in range(3):
        began = time.perf_counter()
        busy.begin()
        q.submit(gemm_cmd(xs, a, b, c, M, N, K, 1))
        q.wait()
        span = time.perf_counter() - began
        torch.cuda.synchronize()
    flushed, rounds, moment = 0, 0, Moment(M, span)
    while flushed < 3 and rounds < 3000:
        rounds += 1
        c.fill_(float("nan"))
        torch.cuda.synchronize()
        busy.begin()
        q.submit(gemm_cmd(xs, a, b, c, M, N, K, 1))
        moment.wait()
        xs.check(p.XQueueSuspend(q.xq, xs.kQueueSuspendFlagSyncHwQueue))
        missing = torch.isnan(c)
        first = plan[0][0] if len(plan) == 2 else 0
        moment.met(missing[:first].any() if first else missing, missing)
        some = bool(missing[first:].any()) and (not bool(missing[:first].any()) if first else not bool(missing.all()))
        xs.check(p.XQueueResume(q.xq, xs.kQueueResumeFlagNone))
        q.wait()
        assert torch.equal(c, want), f"round {rounds}, flushed in the middle: {some}"
        flushed += some
    st = hip_stats(xs, q.hwq)
    q.close()
    print("stats", st, "rounds", rounds, "flushed in the middle", flushed, flush=True)
    assert flushed == 3 and st[1] >= 3 and st[2] >= 3
