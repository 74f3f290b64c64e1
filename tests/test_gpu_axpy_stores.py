"""AXPY where its stores change their way (through the L2 up to 2^24 elements, non-temporal above), and chunks
that end on either side of it, replayed ones too."""
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
