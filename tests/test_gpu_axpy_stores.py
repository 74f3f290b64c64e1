"""AXPY where its stores change their way (through the L2 or non-temporal), chunks that end on either side
of such a size, and arrays that begin off a 128-byte line, replayed ones too."""
import contextlib
import threading

import pytest

pytestmark = pytest.mark.gpu


@contextlib.contextmanager
def queue(xs, torch, level, seed):
    """A queue, at level 2 suspended and resumed at random moments while the block runs."""
    from test_gpu_kernels import Queue
    from test_gpu_preempt import churn
    q, stop = Queue(xs, torch, level, threshold=4, batch=2), threading.Event()
    t = threading.Thread(target=churn, args=(xs, q, stop, seed), daemon=True)
    if level == 2:
        t.start()
    try:
        yield q
    finally:
        stop.set()
        if level == 2:
            t.join()
        q.wait()
        q.close()


def until_replayed(xs, q, level, submit, launches=3):
    """Batches of commands, at level 2 until so many launches were cut short and made again; how many batches it took."""
    from test_gpu_preempt import hip_stats
    batches = 0
    while batches < 200:
        batches += 1
        submit()
        q.wait()
        st = hip_stats(xs, q.hwq)
        if level == 1 or st[1] >= launches:
            break
    print("batches", batches, "stats", st, flush=True)
    assert level == 1 or st[1] >= launches, "too few launches were flushed"
    return batches


@pytest.mark.parametrize("level", [1, 2])
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("n", [(1 << 24) - 1023, 1 << 24, (1 << 24) + 1, (1 << 24) + 1025])
def test_axpy_on_either_side_of_the_limit(xs, gpu, n, offset, level):
    """0.5 x is exact, so the sum is rounded once whoever computes it: bit for bit. The elements around the
    slices stay as they were."""
    from test_gpu_kernels import axpy_cmd
    torch = gpu
    print(f"case axpy-stores n={n} offset={offset} level={level}", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(n)
    x, y = (torch.rand(n + 16, device="cuda", generator=gen) for _ in range(2))
    want, times = y.clone(), 6
    torch.cuda.synchronize()
    with queue(xs, torch, level, n) as q:
        def submit():
            for _ in range(times):
                q.submit(axpy_cmd(xs, 0.5, x[offset:], y[offset:], n, 1 if level == 2 else 0))
        batches = until_replayed(xs, q, level, submit)
    for _ in range(times * batches):
        want[offset:offset + n] += 0.5 * x[offset:offset + n]
    assert torch.equal(y, want)


@pytest.mark.parametrize("grid", ["", "chunk"])
@pytest.mark.parametrize("level", [1, 2])
@pytest.mark.parametrize("x_offset,y_offset", [(0, 1), (3, 31), (1, 32), (5, 16)])
def test_axpy_of_arrays_off_their_lines(xs, gpu, monkeypatch, x_offset, y_offset, level, grid):
    """Chunks begin at the first line of y: arrays that end before it, in it, with the last chunk or a
    few elements from it, and on either side of the sizes from which stores take another way. Bit for bit, and
    nothing around the slices changes."""
    from test_gpu_kernels import axpy_cmd
    torch = gpu
    monkeypatch.setenv("XSCHED_HIP_AXPY_GRID", grid)
    head = -y_offset % 32
    gen = torch.Generator(device="cuda")
    gen.manual_seed(y_offset)
    sizes = {1, head - 1, head, head + 1, head + 4, head + 1023, head + 1024, head + 1025, head + 5 * 1024,
             1 << 20, (1 << 20) + 1, (1 << 21) + 1, 1 << 22, (1 << 22) + 1, 1 << 23, (1 << 23) + head + 1}
    wrong = []
    with queue(xs, torch, level, y_offset) as q:
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
            if not torch.equal(y, want):
                wrong.append(n)
    assert wrong == []


@pytest.mark.parametrize("grid", ["", "chunk"])
@pytest.mark.parametrize("steps", [1, 7])
@pytest.mark.parametrize("n", [(3 << 20) + 5, (1 << 24) - 5])
def test_flushed_slices_are_applied_once(xs, gpu, monkeypatch, n, steps, grid):
    """The elements in front of the first line belong to chunk 0: they are stored behind its look at the preempt word, and
    not again in a replay that finds the chunk done. Chunks of one step and of several, on both grids, with and without stores
    that change their way within the array."""
    from test_gpu_kernels import axpy_cmd
    torch = gpu
    monkeypatch.setenv("XSCHED_HIP_AXPY_GRID", grid)
    monkeypatch.setenv("XSCHED_HIP_AXPY_STEPS", str(steps))
    print(f"case axpy-slices-flushed n={n} steps={steps} grid={grid}", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(n + steps)
    x, y = (torch.rand(n + 80, device="cuda", generator=gen) for _ in range(2))
    want, times, at = y.clone(), 40, 5
    torch.cuda.synchronize()
    with queue(xs, torch, 2, n) as q:
        def submit():
            for _ in range(times):
                q.submit(axpy_cmd(xs, 0.5, x[at:], y[at:], n, 1))
        batches = until_replayed(xs, q, 2, submit, launches=8)
    for _ in range(times * batches):
        want[at:at + n] += 0.5 * x[at:at + n]
    assert torch.equal(y[:at + 32], want[:at + 32])
    assert torch.equal(y, want)
