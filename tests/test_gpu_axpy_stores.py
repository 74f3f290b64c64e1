"""AXPY where its stores change their way (through the L2 or non-temporal), chunks that end on either side
of such a size, and arrays that begin off a 128-byte line, replayed ones too."""
import threading

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level", [1, 2])
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("n", [(1 << 24) - 1023, 1 << 24, (1 << 24) + 1, (1 << 24) + 1025])
def test_axpy_on_either_side_of_the_limit(xs, gpu, n, offset, level):
    """0.5 x is exact, so the sum is rounded once whoever computes it: bit for bit. The elements around the
    slices stay as they were."""
    from test_gpu_kernels import Queue, axpy_cmd
    from test_gpu_preempt import churn
    torch = gpu
    print(f"case axpy-stores n={n} offset={offset} level={level}", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(n)
    x, y = (torch.rand(n + 16, device="cuda", generator=gen) for _ in range(2))
    want = y.clone()
    times = 6
    for _ in range(times):
        want[offset:offset + n] += 0.5 * x[offset:offset + n]
    torch.cuda.synchronize()
    q, stop = Queue(xs, torch, level), threading.Event()
    t = threading.Thread(target=churn, args=(xs, q, stop, n))
    if level == 2:
        t.start()
    for _ in range(times):
        q.submit(axpy_cmd(xs, 0.5, x[offset:], y[offset:], n, 1 if level == 2 else 0))
    q.wait()
    if level == 2:
        stop.set()
        t.join()
    q.close()
    assert torch.equal(y, want)


@pytest.mark.parametrize("grid", ["", "chunk"])
@pytest.mark.parametrize("level", [1, 2])
@pytest.mark.parametrize("x_offset,y_offset", [(0, 1), (3, 31), (1, 32), (5, 16)])
def test_axpy_of_arrays_off_their_lines(xs, gpu, monkeypatch, x_offset, y_offset, level, grid):
    """Chunks begin at the first line of y: arrays that end before it, in it, with the last chunk or a
    few elements from it, and on either side of the sizes from which stores take another way. Bit for bit, and
    nothing around the slices changes."""
    from test_gpu_kernels import Queue, axpy_cmd
    from test_gpu_preempt import churn
    torch = gpu
    monkeypatch.setenv("XSCHED_HIP_AXPY_GRID", grid)
    head = -y_offset % 32
    gen = torch.Generator(device="cuda")
    gen.manual_seed(y_offset)
    q, stop = Queue(xs, torch, level), threading.Event()
    t = threading.Thread(target=churn, args=(xs, q, stop, y_offset))
    if level == 2:
        t.start()
    sizes = {1, head - 1, head, head + 1, head + 4, head + 1023, head + 1024, head + 1025, head + 5 * 1024,
             1 << 22, (1 << 22) + 1, 1 << 23, (1 << 23) + head + 1}
    for n in sorted(n for n in sizes if n > 0):
        print(f"case axpy-lines n={n} x_offset={x_offset} y_offset={y_offset} level={level} grid={grid}", flush=True)
        x, y = (torch.rand(n + 80, device="cuda", generator=gen) for _ in range(2))
        assert y.data_ptr() % 128 == 0
        want = y.clone()
        for _ in range(3):
            want[y_offset:y_offset + n] += 0.5 * x[x_offset:x_offset + n]
        torch.cuda.synchronize()
        for _ in range(3):
            q.submit(axpy_cmd(xs, 0.5, x[x_offset:], y[y_offset:], n, 1 if level == 2 else 0))
        q.wait()
        assert torch.equal(y, want), n
    if level == 2:
        stop.set()
        t.join()
    q.close()
