"""Performance cases of the command queue and its guarded kernels.

A case is a plain dict; ``prepare(case, seed)`` makes what a program has in hand (device arrays),
``run(state)`` takes ONE pass through the public entry points: commands are created, submitted to
their XQueues and waited for, as a program that needs the results does. Queues belong to the
program, not to its data: they are created once per process and used for whatever comes.

Kinds of cases:
    axpy  y = 0.5 x + y in place over n floats, ``commands`` times on one queue
    gemm  C = A B, bf16, M x N x K
    hist  bins[key] += 1 over n int32 keys; on ``queues`` queues side by side (arrays of their own),
          or (``direct``) with the call that takes a stream instead of a queue
    preempt  two GEMMs of bg^3 on a low-priority queue, then one of fg^3 on a high-priority one:
          the scheduler flushes the running GEMM, runs the short one and resumes
Fields shared by them: ``level`` is the preemption level of the queue (1: commands run to their
end, 2: guarded kernels that can be flushed); ``offset`` is how many elements behind an aligned
address the arrays start (a slice of a larger array).
"""
import ctypes
import math

import torch

import xsched_amd as xs

ALPHA = 0.5
ZIPF_S = 1.1
HIST_BINS = 65536


def listed():
    return [
        # The smallest command a latency-bound foreground queue gets: all of it is launch and wait.
        dict(name="axpy_64k", kind="axpy", n=1 << 16, offset=0, commands=1, level=1),
        # The foreground command of the streaming configuration.
        dict(name="axpy_4m", kind="axpy", n=1 << 22, offset=0, commands=1, level=1),
        # A slice of a larger array: 4-byte aligned start, a length that is no multiple of anything.
        dict(name="axpy_16m_slice", kind="axpy", n=(1 << 24) - 5, offset=1, commands=1, level=2),
        # The background of the streaming configuration: long arrays back to back, flushable.
        dict(name="axpy_256m", kind="axpy", n=1 << 28, offset=0, commands=2, level=2),
        # The foreground command of the matrix configuration.
        dict(name="gemm_1k", kind="gemm", M=1024, N=1024, K=1024, offset=0, level=2),
        # The matrix command of the mixed configuration.
        dict(name="gemm_2k", kind="gemm", M=2048, N=2048, K=2048, offset=0, level=2),
        # The background of the matrix configuration.
        dict(name="gemm_8k", kind="gemm", M=8192, N=8192, K=8192, offset=0, level=2),
        # Odd sizes in every dimension: no row starts on a 16-byte boundary.
        dict(name="gemm_odd", kind="gemm", M=2000, N=1999, K=2047, offset=0, level=2),
        # The foreground command of the histogram configuration.
        dict(name="hist_1m", kind="hist", n=1 << 20, bins=HIST_BINS, zipf=True, offset=0, queues=1, direct=False, level=2),
        # A histogram of few bins over evenly spread keys, enqueued on the program's own stream.
        dict(name="hist_16m_1000_bins", kind="hist", n=(1 << 24) + 77, bins=1000, zipf=False, offset=0, queues=1, direct=True, level=1),
        # The background of the histogram configuration: four queues side by side.
        dict(name="hist_4x64m", kind="hist", n=1 << 26, bins=HIST_BINS, zipf=True, offset=0, queues=4, direct=False, level=2),
        # What the library is for: a short command arrives while long ones run.
        dict(name="preempt_gemm", kind="preempt", bg=4096, fg=1024, level=2),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["axpy"] * 6 + ["gemm"] * 7 + ["hist"] * 6 + ["preempt"])
    level = rng.choice([1, 2, 2])
    if kind == "axpy":
        n = _log_uniform(rng, 1 << 12, 1 << 28)
        if rng.random() < 0.4:
            n = max(1024, n // 1024 * 1024)
        return dict(kind=kind, n=n, offset=rng.choice([0, 0, 0, 1, 2, 3]), commands=rng.choice([1, 1, 2]), level=level)
    if kind == "gemm":
        M, N, K = (_log_uniform(rng, 64, 8192) for _ in range(3))
        offset = 0
        shape = rng.random()

        def whole(v, unit):
            return max(unit, v // unit * unit)
        if shape < 0.4:       # everything a multiple of the tiles
            M, N, K = whole(M, 128), whole(N, 128), whole(K, 64)
        elif shape < 0.6:     # a ragged batch dimension
            N, K = whole(N, 128), whole(K, 64)
        elif shape < 0.8:     # rows that start on 16-byte boundaries
            M, N, K = whole(M, 8), whole(N, 8), whole(K, 8)
        else:
            offset = rng.choice([0, 0, 1])
        return dict(kind=kind, M=M, N=N, K=K, offset=offset, level=level)
    if kind == "hist":
        n = _log_uniform(rng, 1 << 12, 1 << 26)
        if rng.random() < 0.3:
            n = n // 4096 * 4096
        bins = rng.choice([HIST_BINS, HIST_BINS, _log_uniform(rng, 16, HIST_BINS)])
        direct = rng.random() < 0.25
        return dict(kind=kind, n=n, bins=bins, zipf=rng.random() < 0.6, offset=rng.choice([0, 0, 0, 1]),
                    queues=1 if direct else rng.choice([1, 1, 2, 4]), direct=direct, level=1 if direct else level)
    return dict(kind=kind, bg=128 * rng.randint(16, 40), fg=128 * rng.randint(4, 12), level=2)


# ---- the program's queues -------------------------------------------------------------------

_queues = {}


def _queue(role, level):
    """The XQueue for one role of this program ("fg" outranks "bg0" .. "bg3"), made at first use."""
    key = (role, level)
    if key not in _queues:
        p = xs.preempt()
        if not _queues:
            xs.check(p.XHintSetScheduler(xs.kSchedulerLocal, xs.kPolicyHighestPriorityFirst))
        stream = torch.cuda.Stream()
        xq = xs.xqueue_create(xs.hip_queue_create(stream.cuda_stream), level)
        # background: one command running, one behind it; foreground: the window never fills
        xs.check(p.XQueueSetLaunchConfig(xq, *((8, 4) if role == "fg" else (2, 1))))
        xs.check(p.XHintPriority(xq, 1 if role == "fg" else 0))
        _queues[key] = (xq, stream)
    return _queues[key][0]


# ---- inputs ---------------------------------------------------------------------------------

_zipf_cdf = {}


def _keys(gen, n, bins, zipf, offset):
    if not zipf:
        return torch.randint(0, bins, (n + offset,), dtype=torch.int32, device="cuda", generator=gen)[offset:]
    if bins not in _zipf_cdf:
        w = torch.arange(1, bins + 1, dtype=torch.float64, device="cuda").pow(-ZIPF_S).cumsum(0)
        _zipf_cdf[bins] = (w / w[-1]).float()
    u = torch.rand(n + offset, device="cuda", generator=gen)
    keys = torch.searchsorted(_zipf_cdf[bins], u, right=True, out_int32=True)
    return keys.clamp_(max=bins - 1)[offset:]


def _bf16(gen, rows, cols, offset):
    flat = torch.randn(rows * cols + offset, device="cuda", generator=gen).to(torch.bfloat16)
    return flat[offset:].view(rows, cols)


def _gemm_arrays(gen, M, N, K, offset):
    c = torch.zeros(M * N + offset, dtype=torch.bfloat16, device="cuda")[offset:].view(M, N)
    return _bf16(gen, M, K, offset), _bf16(gen, K, N, offset), c


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind, level = case["kind"], case["level"]
    s = dict(case)
    if kind == "axpy":
        n, off = case["n"], case["offset"]
        s["xq"] = _queue("fg" if level == 1 else "bg0", level)
        s["x"], s["y"] = (torch.rand(n + off, device="cuda", generator=gen).mul_(2).sub_(1)[off:] for _ in range(2))
    elif kind == "gemm":
        s["xq"] = _queue("fg" if level == 1 else "bg0", level)
        s["abc"] = _gemm_arrays(gen, case["M"], case["N"], case["K"], case["offset"])
    elif kind == "hist":
        s["xqs"] = [] if case["direct"] else [_queue("bg%d" % q, level) for q in range(case["queues"])]
        s["keys"] = [_keys(gen, case["n"], case["bins"], case["zipf"], case["offset"]) for _ in range(case["queues"])]
        s["counts"] = [torch.zeros(case["bins"], dtype=torch.int32, device="cuda") for _ in range(case["queues"])]
    else:
        s["bg_xq"], s["fg_xq"] = _queue("bg0", level), _queue("fg", level)
        s["bg_abc"] = [_gemm_arrays(gen, case["bg"], case["bg"], case["bg"], 0) for _ in range(2)]
        s["fg_abc"] = _gemm_arrays(gen, case["fg"], case["fg"], case["fg"], 0)
    return s


# ---- one pass -------------------------------------------------------------------------------

def _submit(xq, create, *args):
    cmd = ctypes.c_uint64()
    xs.check(create(ctypes.byref(cmd), *args))
    xs.check(xs.preempt().XQueueSubmit(xq, cmd.value))


def _submit_gemm(xq, abc, guard):
    a, b, c = abc
    _submit(xq, xs.halhip().HipGemmBf16CommandCreate, a.data_ptr(), b.data_ptr(), c.data_ptr(),
            a.shape[0], b.shape[1], a.shape[1], guard)


def _wait(xq):
    xs.check(xs.preempt().XQueueWaitAll(xq))


def run(s):
    kind = s["kind"]
    guard = 0 if s["level"] == 1 else 1
    if kind == "axpy":
        for _ in range(s["commands"]):
            _submit(s["xq"], xs.halhip().HipAxpyCommandCreate, ALPHA, s["x"].data_ptr(), s["y"].data_ptr(), s["n"], guard)
        _wait(s["xq"])
        return s["y"]
    if kind == "gemm":
        _submit_gemm(s["xq"], s["abc"], guard)
        _wait(s["xq"])
        return s["abc"][2]
    if kind == "hist":
        if s["direct"]:
            xs.check(xs.halhip().HipHistogramLaunchNoAlloc(torch.cuda.current_stream().cuda_stream, s["keys"][0].data_ptr(),
                                                           s["n"], s["counts"][0].data_ptr(), s["bins"]))
            return s["counts"]
        for xq, keys, counts in zip(s["xqs"], s["keys"], s["counts"]):
            _submit(xq, xs.halhip().HipHistogramCommandCreate, keys.data_ptr(), s["n"], counts.data_ptr(), s["bins"], guard)
        for xq in s["xqs"]:
            _wait(xq)
        return s["counts"]
    for abc in s["bg_abc"]:
        _submit_gemm(s["bg_xq"], abc, guard)
    _submit_gemm(s["fg_xq"], s["fg_abc"], guard)
    _wait(s["fg_xq"])
    _wait(s["bg_xq"])
    return [s["fg_abc"][2]] + [abc[2] for abc in s["bg_abc"]]


# ---- what a pass cannot do without ----------------------------------------------------------

def _gemm_work(M, N, K):
    return 2 * (M * K + K * N + M * N), 2 * M * N * K


def work(case):
    kind = case["kind"]
    if kind == "axpy":   # x and y in, y out
        return dict(bytes=12 * case["n"] * case["commands"], flops=2 * case["n"] * case["commands"])
    if kind == "gemm":
        b, f = _gemm_work(case["M"], case["N"], case["K"])
        return dict(bytes=b, flops=f)
    if kind == "hist":   # the keys in, the bins in and out
        return dict(bytes=case["queues"] * (4 * case["n"] + 8 * case["bins"]), flops=0)
    (b0, f0), (b1, f1) = (_gemm_work(case[k], case[k], case[k]) for k in ("bg", "fg"))
    return dict(bytes=2 * b0 + b1, flops=2 * f0 + f1)


def tolerance(case):
    if case["kind"] in ("axpy", "hist"):   # one rounding per element; whole numbers
        return "exact"
    # bf16 results of fp32 sums: 1.7e-3 (2-norm) and 3.9e-3 (largest) off the product in 64 bits,
    # which is the rounding of the result alone
    return {"rel": 6.6e-3, "max": 1.6e-2}
