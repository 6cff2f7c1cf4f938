"""A small transfer does not wait for another solver's large ones: each large download
holds the staging slots for its whole length, and a small one has slots of its own."""
import threading
import time

import numpy as np
import pytest

import nekwave_amd as nw

pytestmark = pytest.mark.gpu


def _solver(n1, nel, precision="fp32"):
    m = nw.Mesh(n1)
    m.createBoxMesh(*nel, 0, 1, 0, 1, 0, 1)
    s = nw.DgSolver(precision=precision)
    s.initialize(m, 1.0)
    s.uploadState(np.ones(6 * m.getTotalPoints()))
    return m, s


def _alone(f, n):
    t = []
    for _ in range(n):
        t0 = time.perf_counter()
        f()
        t.append(time.perf_counter() - t0)
    return float(np.median(t))


def test_small_transfers_pass_a_large_one():
    mb, big = _solver(8, (24, 24, 24))  # 340 MB of host array
    ms, small = _solver(3, (4, 4, 4))   # 83 kB
    small.setProbes(ms, [[0.3, 0.4, 0.5]], capacity=8)
    host = np.zeros(6 * mb.getTotalPoints())
    out = np.zeros(6 * ms.getTotalPoints())

    def few():
        small.downloadState(out)
        small.uploadState(out)
        small.sampleProbes()
        assert small.probeHistory().shape == (1, 1, 6)

    one = _alone(lambda: big.downloadState(host), 5)
    _alone(few, 5)
    stop = threading.Event()

    def many():
        while not stop.is_set():
            big.downloadState(host)

    th = threading.Thread(target=many)
    th.start()
    try:
        time.sleep(0.02)
        beside = _alone(few, 21)
    finally:
        stop.set()
        th.join()
    assert np.array_equal(out, np.ones(out.size)) and np.array_equal(host, np.ones(host.size))
    # three transfers that each waited for the one in hand would take one to three of them
    assert beside < 0.5 * one, (beside, one)
    big.finalize()
    small.finalize()
