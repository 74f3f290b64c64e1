"""A queue that its application and the scheduler's rounds suspend and resume at the same time
never stays paused behind the last resume (tests/suspend_race_driver.cpp; with Suspend() and
Resume() free to interleave it got stuck within 170 of its rounds)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "xsched_amd", "lib")


def test_application_and_scheduler_suspend_the_same_queue(xs, tmp_path):
    if not os.path.exists(os.path.join(LIB, "libhalhost.so")):
        pytest.skip("libraries not built")
    exe = str(tmp_path / "suspend_race")
    subprocess.run(["g++", "-std=c++20", "-O2", "-I", os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "suspend_race_driver.cpp"), "-o", exe,
                    "-L", LIB, "-Wl,-rpath," + LIB, "-lhalhost", "-lpreempt", "-pthread"], check=True)
    out = subprocess.run([exe, "3000"], capture_output=True, text=True, timeout=110, env=dict(os.environ, XLOG_LEVEL="WARN"))
    assert out.returncode == 0, out.stdout + out.stderr
