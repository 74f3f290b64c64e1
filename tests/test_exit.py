"""A process that ends with its queues alive: the scheduler still takes events while the exit handlers run,
and must not use anything that was destroyed before. Freed memory is overwritten by the C library
(MALLOC_PERTURB_, without the per-thread caches, which keep it), so that a use of it shows. CPU only."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
import time
from ctypes import byref, c_uint64
import xsched_amd as xs
p, h = xs.preempt(), xs.halhost()
xq = xs.xqueue_create(xs.host_queue_create())
busy = xs.HostKernelFn(lambda *args: time.sleep(0.05))
cmd = c_uint64()
xs.check(h.HostKernelCommandCreate(byref(cmd), busy, None, 1, 0))
xs.check(p.XQueueSubmit(xq, cmd.value))
xs.check(p.XQueueWaitAll(xq))
print("end of the program", flush=True)
"""


@pytest.mark.parametrize("policy", ["HPF", "CFS"])
def test_process_ends_cleanly_with_its_queues_alive(policy):
    env = dict(os.environ, XSCHED_SCHEDULER="LCL", XSCHED_POLICY=policy, XLOG_LEVEL="ERRO", PYTHONPATH=ROOT,
               MALLOC_PERTURB_="165", GLIBC_TUNABLES="glibc.malloc.tcache_count=0")
    run = subprocess.run([sys.executable, "-c", PROGRAM], env=env, capture_output=True, text=True, timeout=120)
    assert run.stdout.strip() == "end of the program"
    assert run.returncode == 0, (run.returncode, run.stderr[-2000:])
