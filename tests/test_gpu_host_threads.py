"""A native call gives the interpreter's lock back while it takes device memory and launches: another Python thread runs
meanwhile.  With a switch interval of minutes a thread gets the lock only where its holder gives it up."""
import sys
import threading
import time

import pytest
import torch

from gpu_util import note
from var_q_amd import PackedKVCache, ops

pytestmark = pytest.mark.gpu


def _ticks_during(work):
    ticks, stop = [0], threading.Event()

    def ticker():
        while not stop.is_set():
            ticks[0] += 1
            time.sleep(1e-4)

    other, before = threading.Thread(target=ticker), sys.getswitchinterval()
    sys.setswitchinterval(600)
    try:
        other.start()
        while ticks[0] < 3:
            time.sleep(1e-3)
        first = ticks[0]
        work()
        return ticks[0] - first
    finally:
        sys.setswitchinterval(before)
        stop.set()
        other.join()


def test_another_thread_runs_during_a_call(dev):
    note('interpreter lock: fresh allocations')
    words = torch.zeros(1 << 27, 1, dtype=torch.int32, device=dev)
    ops.unpack(words[:1], 4, 8)
    torch.cuda.synchronize()
    keep = []

    def calls():       # 512 MiB that no call before has given back, 24 times: each takes its memory from the device
        for _ in range(24):
            keep.append(ops.unpack(words, 4, 8))

    assert _ticks_during(calls) > 0
    del keep
    torch.cuda.empty_cache()


def test_threads_on_streams_of_their_own(dev):
    """Four threads, a cache and a stream each: every result is that of the same calls in one thread."""
    note('interpreter lock: four threads')

    def inputs(i):
        gen = torch.Generator(device=dev).manual_seed(i)
        return [tuple(torch.randn(2, 4, n, 64, device=dev, generator=gen).bfloat16() for _ in range(3)) for n in (1, 9, 64, 100)]

    def schedule(i, steps):
        cache = PackedKVCache(2, 4, 174, 64, 4 if i % 2 else [2, 4, 8, 4], 32, dev)
        outs = []
        for q, k, v in steps:
            cache.append(k, v)
            outs.append(cache.attend(q, 0.125))
        return outs

    steps = [inputs(i) for i in range(4)]
    want = [schedule(i, s) for i, s in enumerate(steps)]
    torch.cuda.synchronize()
    got = [None] * 4

    def run(i):
        with torch.cuda.stream(torch.cuda.Stream(dev)):
            for _ in range(20):
                got[i] = schedule(i, steps[i])

    threads = [threading.Thread(target=run, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for a, b in zip(want, got):
        assert all(torch.equal(x, y) for x, y in zip(a, b))
