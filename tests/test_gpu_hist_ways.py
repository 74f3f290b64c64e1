"""GPU parity of the histogram where it changes its ways by itself: few keys, one kernel or two,
whole-word, half-word and byte counters, and key arrays at any multiple of four bytes."""
import threading

import numpy as np
import pytest

import oracle
from test_gpu_kernels import Queue, hist_cmd
from test_gpu_preempt import churn, hip_stats

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_bins", [1, 255, 256, 257, 16383, 16384, 16385, 32768, 32769, 49153, 65536])
@pytest.mark.parametrize("n,offset", [(1, 0), (1023, 1), (1024, 0), (1025, 3), (1 << 16, 0), ((1 << 16) + 1, 2), (1 << 18, 1),
                                      ((1 << 21) + 4099, 0)])
@pytest.mark.parametrize("level,guard", [(1, 0), (2, 1)])
def test_histogram_ways_by_size_and_bins(xs, gpu, n, offset, n_bins, level, guard):
    """Counts are whole numbers: bit for bit the oracle's. One key in eight is the last bin (it
    fills a byte counter several times over from 2048 keys of a group on), a few lie outside
    the bins and count nowhere; twice, since bins are added to."""
    torch = gpu
    print(f"case hist-ways n={n} offset={offset} bins={n_bins} level={level} guard={guard}", flush=True)
    rng = np.random.default_rng(n + n_bins)
    keys_h = rng.integers(0, n_bins, n).astype(np.int32)
    keys_h[rng.random(n) < 0.125] = n_bins - 1
    outside = rng.random(n) < 0.01
    keys_h[outside] = rng.choice(np.array([-1, n_bins, n_bins + 16384, 1 << 30], np.int32), int(outside.sum()))
    keys = torch.from_numpy(np.concatenate([np.zeros(offset, np.int32), keys_h])).cuda()[offset:]
    bins = torch.zeros(n_bins + 1, dtype=torch.int32, device="cuda")
    q = Queue(xs, torch, level)
    for _ in range(2):
        q.submit(hist_cmd(xs, keys, n, bins, n_bins, guard))
    q.wait()
    got = bins.cpu().numpy().view(np.uint32)
    q.close()
    want = oracle.histogram(keys_h[~outside], n_bins)
    assert np.array_equal(got[:n_bins], 2 * want)
    assert got[n_bins] == 0, "wrote beyond the bins array"


@pytest.mark.parametrize("n_bins", [254, 255, 256, 257, 4032, 4033, 4096, 4097, 65536])
@pytest.mark.parametrize("n", [(1 << 16) + 1, (1 << 24) + 5, (1 << 25) + 5])
def test_histogram_counters_of_the_hot_bins(xs, gpu, n, n_bins):
    """Around the number of bins from which the hot ones have fewer counters, with the hottest bin
    in every second key, and around the length from which work-groups share a compute unit: on
    two queues at once, so that they do. Whole numbers: bit for bit the oracle's."""
    torch = gpu
    print(f"case hist-hot n={n} bins={n_bins}", flush=True)
    rng = np.random.default_rng(n + n_bins)
    keys_h = rng.integers(0, n_bins, n).astype(np.int32)
    keys_h[::2] = rng.integers(0, 2) * 253
    keys_h[1::64] = 254          # no bin where n_bins is 254
    keys = torch.from_numpy(keys_h).cuda()
    bins = [torch.zeros(n_bins + 1, dtype=torch.int32, device="cuda") for _ in range(2)]
    queues = [Queue(xs, torch, 2) for _ in bins]
    for q, b in zip(queues, bins):
        q.submit(hist_cmd(xs, keys, n, b, n_bins, 1))
    for q in queues:
        q.wait()
    got = [b.cpu().numpy().view(np.uint32) for b in bins]
    for q in queues:
        q.close()
    want = oracle.histogram(keys_h[keys_h < n_bins], n_bins)
    for g in got:
        assert np.array_equal(g[:n_bins], want)
        assert g[n_bins] == 0, "wrote beyond the bins array"


def _command_us(xs, torch, keys, n_bins):
    """Least time of a histogram command of several, in us."""
    bins = torch.zeros(n_bins, dtype=torch.int32, device="cuda")
    stream = torch.cuda.current_stream()
    best = float("inf")
    for _ in range(7):
        start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        start.record()
        for _ in range(4):
            xs.check(xs.halhip().HipHistogramLaunchNoAlloc(stream.cuda_stream, keys.data_ptr(), keys.numel(), bins.data_ptr(), n_bins))
        end.record()
        torch.cuda.synchronize()
        best = min(best, start.elapsed_time(end) * 250)
    return best


def test_histogram_of_256_bins_counts_the_last_bin_like_the_others(xs, gpu):
    """Bytes that are all 255 (an image's white) took 5 times as long as bytes that are all 0: one
    counter for all lanes of a work-group."""
    torch = gpu
    print("case hist-256", flush=True)
    first, last = (_command_us(xs, torch, torch.full((1 << 25,), key, dtype=torch.int32, device="cuda"), 256) for key in (0, 255))
    print("us", first, last, flush=True)
    assert last < 2 * first


def test_histogram_of_one_key_outside_the_warm_bins(xs, gpu):
    """Equal keys outside the first 255 of 65536 bins overflow their counters: counted, and counted again,
    within 4 times what equal keys of bin 0 take (6.5 times before runs of one key were added together)."""
    torch = gpu
    print("case hist-one-key", flush=True)
    first, cold = (_command_us(xs, torch, torch.full((1 << 24,), key, dtype=torch.int32, device="cuda"), 65536) for key in (0, 300))
    print("us", first, cold, flush=True)
    assert cold < 4 * first


@pytest.mark.parametrize("n,offset", [(4096, 0), (8192, 1), ((1 << 16) + 1, 0), ((1 << 18) + 4095, 3), ((1 << 22) + 5, 0)])
@pytest.mark.parametrize("n_bins", [1000, 20000, 40000, 65536])
@pytest.mark.parametrize("shape", ["constant", "sorted", "descending", "runs", "ends"])
def test_histogram_of_runs(xs, gpu, n, offset, n_bins, shape):
    """Runs of one key of every kind, with keys outside the bins among them: bit for bit the oracle's."""
    torch = gpu
    print(f"case hist-runs n={n} offset={offset} bins={n_bins} {shape}", flush=True)
    rng = np.random.default_rng(n + n_bins)
    if shape == "constant":
        keys_h = np.full(n, n_bins - 300, np.int32)
    elif shape == "sorted":
        keys_h = np.sort(rng.integers(-3, n_bins + 3, n)).astype(np.int32)
    elif shape == "descending":
        keys_h = np.sort(rng.integers(0, n_bins, n))[::-1].astype(np.int32)
    elif shape == "runs":
        keys_h = np.repeat(rng.integers(-1, n_bins + 1, n // 7 + 1), rng.integers(1, 600, n // 7 + 1))[:n].astype(np.int32)
        keys_h = np.resize(keys_h, n)
    else:   # two keys far apart: the quarters of the bins between them are empty
        keys_h = np.where(np.arange(n) // 512 % 2 == 0, 300, n_bins - 1).astype(np.int32)
    keys = torch.from_numpy(np.concatenate([np.zeros(offset, np.int32), keys_h])).cuda()[offset:]
    bins = torch.zeros(n_bins + 1, dtype=torch.int32, device="cuda")
    q = Queue(xs, torch, 2)
    for _ in range(2):
        q.submit(hist_cmd(xs, keys, n, bins, n_bins, 1))
    q.wait()
    got = bins.cpu().numpy().view(np.uint32)
    q.close()
    want = oracle.histogram(np.ascontiguousarray(keys_h[(keys_h >= 0) & (keys_h < n_bins)]), n_bins)
    assert np.array_equal(got[:n_bins], 2 * want)
    assert got[n_bins] == 0, "wrote beyond the bins array"


@pytest.mark.parametrize("n_bins,hot", [(20000, [300]), (20000, [300, 300 + 16384]), (32768, [32767]), (32768, [16383, 32767]),
                                        (65536, [300, 300 + 16384, 300 + 49152]), (16384, [300]), (16384, [255, 16383]), (5000, [4999])])
@pytest.mark.parametrize("way", ["sweep", "merge"])
@pytest.mark.parametrize("n", [1 << 18, (1 << 19) + 70001])
def test_histogram_counters_that_take_more_than_16_bits(xs, gpu, monkeypatch, n_bins, hot, way, n):
    """Work-groups of 2^18 keys with one, two or three bins outside the warm ones, in one word where a word holds
    several, that take more than 2^16 keys of a group each: half words (and bytes) overflow and are recounted, whole
    words hold them, through both ways of merging. Whole numbers: bit for bit the oracle's."""
    torch = gpu
    print(f"case hist-16bit n={n} bins={n_bins} hot={hot} {way}", flush=True)
    monkeypatch.setenv("XSCHED_HIP_HIST_MIN_CHUNK", str(1 << 18))
    monkeypatch.setenv("XSCHED_HIP_HIST_MERGE_MIN_KEYS", "1" if way == "merge" else str(1 << 40))
    rng = np.random.default_rng(n_bins + len(hot))
    keys_h = rng.integers(0, n_bins, n).astype(np.int32)
    hot_at = rng.random(n) < 0.9
    keys_h[hot_at] = rng.choice(np.array(hot, np.int32), int(hot_at.sum()))
    keys = torch.from_numpy(keys_h).cuda()
    bins = torch.zeros(n_bins + 1, dtype=torch.int32, device="cuda")
    q = Queue(xs, torch, 2)
    q.submit(hist_cmd(xs, keys, n, bins, n_bins, 1))
    q.wait()
    got = bins.cpu().numpy().view(np.uint32)
    q.close()
    want = oracle.histogram(keys_h, n_bins)
    assert min(int(np.sum(keys_h[:1 << 18] == h)) for h in hot) > 1 << 16
    assert np.array_equal(got[:n_bins], want)
    assert got[n_bins] == 0, "wrote beyond the bins array"


@pytest.mark.parametrize("n,n_bins", [((1 << 16) - 3, 65536), (1 << 16, 20000)])
def test_few_keys_flushed_and_replayed(xs, gpu, n, n_bins):
    """The kernel for few keys over many bins, suspended and resumed until launches of it have been
    replayed a few times: every command counts once. A command takes some 5 us, so they come in rounds."""
    torch = gpu
    print(f"case few-keys-flush n={n} bins={n_bins}", flush=True)
    rng = np.random.default_rng(n)
    keys_h = rng.integers(0, n_bins, n).astype(np.int32)
    keys = torch.from_numpy(keys_h).cuda()
    bins = torch.zeros(n_bins, dtype=torch.int32, device="cuda")
    q = Queue(xs, torch, level=2, threshold=4, batch=2)
    stop = threading.Event()
    t = threading.Thread(target=churn, args=(xs, q, stop, 5))
    t.start()
    times = 0
    while times < 20000:
        for _ in range(100):
            q.submit(hist_cmd(xs, keys, n, bins, n_bins, 1))
        times += 100
        st = hip_stats(xs, q.hwq)
        if st[1] >= 5 and st[2] >= 5:
            break
    stop.set()
    t.join()
    q.wait()
    st = hip_stats(xs, q.hwq)
    got = bins.cpu().numpy().view(np.uint32)
    q.close()
    print("stats", st, "commands", times, flush=True)
    assert st[1] >= 5 and st[2] >= 5, "too few launches were replayed"
    assert np.array_equal(got.astype(np.uint64), (oracle.histogram(keys_h, n_bins).astype(np.uint64) * times) & 0xFFFFFFFF)
