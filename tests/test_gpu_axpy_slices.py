"""GPU parity of AXPY on slices of larger arrays: the vector kernels at every multiple of four
bytes, at lengths around the chunk of a wave and around the borders where the number of
long-lived waves per compute unit changes (2^22 and 2^24 elements)."""
import numpy as np
import pytest

import oracle
from test_gpu_kernels import Queue, axpy_cmd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 4, 1023, 1025, 4099, (1 << 22) + 1, (1 << 24) + 1025])
@pytest.mark.parametrize("x_off,y_off", [(1, 0), (0, 3), (1, 2), (2, 2)])
@pytest.mark.parametrize("level,guard", [(1, 0), (2, 1)])
def test_axpy_on_slices(xs, gpu, n, x_off, y_off, level, guard):
    torch = gpu
    print(f"case axpy-slice n={n} x+{x_off} y+{y_off} level={level} guard={guard}", flush=True)
    x_h = oracle.fill_uniform(31, 1, 0, n + 4)
    y_h = oracle.fill_uniform(31, 2, 0, n + 8)
    x, y = torch.from_numpy(x_h).cuda(), torch.from_numpy(y_h.copy()).cuda()
    q = Queue(xs, torch, level)
    q.submit(axpy_cmd(xs, 0.3337, x[x_off:], y[y_off:], n, guard))
    q.wait()
    got = y.cpu().numpy()
    q.close()
    want = y_h.copy()
    want[y_off:y_off + n] = oracle.axpy(np.float32(0.3337), x_h[x_off:x_off + n], y_h[y_off:y_off + n])
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
