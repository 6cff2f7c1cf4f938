"""Which launches run: a mesh that fits on chip takes resident launches where those are the
faster route, and every one of them completes, from one workgroup per CU up to the largest
mesh the launcher places (an overestimate would show as launches that give up, whose steps run again by stage
launches with the same result), and one that gives up is counted as such."""
import fcntl
import glob
import threading
import time

import numpy as np
import pytest

import nekwave_amd as nw

pytestmark = pytest.mark.gpu


def _solver(m, precision, seed=7, **kw):
    s = nw.DgSolver(precision=precision, **kw)
    s.initialize(m, 1.0)
    s.uploadState(np.random.default_rng(seed).standard_normal(6 * m.getTotalPoints()))
    return s


def _box(n1, nel, jitter=0.1):
    m = nw.Mesh(n1)
    m.createBoxMesh(*nel, 0, 1, 0, 1, 0, 1, True, False, False, jitter=jitter, seed=3)
    return m


@pytest.mark.parametrize("precision", ["fp64", "fp32", "fp32_k64"])
@pytest.mark.parametrize("n1", range(2, 10))
def test_resident_launches_complete_up_to_the_largest_mesh(n1, precision):
    for jitter in (0.0, 0.1):
        for k in (1, 2, 3, 4, 6, 8, 12, 16, 20, 24, 32, 36, 40, 44, 48, 64, 72, 80, 88, 96, 128):  # multiples of 256 workgroups
            m = _box(n1, (16, 16, k), jitter)
            s = _solver(m, precision)
            # enough stages for every element to wait on every other: with a few, workgroups
            # that were not placed at first would find room when others are through
            s.run(0.1 * m.computeMinNodeDistance(), 40)
            done, lost = s.residentLaunches()
            s.finalize()
            assert lost == 0, (jitter, k)
            assert done > 0 or k > 1 or (n1, precision) == (2, "fp64"), (jitter, k)
            if done == 0:  # does not fit, or stage launches are faster
                break


def test_stage_launches_are_not_counted_as_resident(monkeypatch):
    m = _box(5, (4, 3, 2))
    for kw in ({"tile_option": 0}, {"precision": "fp64", "pipeline": "plain"}):
        s = _solver(m, **{"precision": "fp32", **kw})
        s.run(1e-3, 3)
        assert s.residentLaunches() == (0, 0)
        s.finalize()
    monkeypatch.setenv("NW_RESIDENT", "0")
    s = _solver(m, "fp32")
    s.run(1e-3, 3)
    assert s.residentLaunches() == (0, 0)
    s.finalize()


# stage launches are the faster route from some size on, well below what fits (n1 < 4: an
# element fills a part of a wave; jittered or FP64: kernels that spill registers)
@pytest.mark.parametrize("n1,precision,jitter,few,many", [
    (2, "fp64", 0.0, 0, 1), (2, "fp32", 0.1, 10, 12), (3, "fp64", 0.0, 5, 6), (3, "fp32_k64", 0.1, 8, 9),
    (4, "fp32", 0.1, 44, 52), (4, "fp64", 0.1, 16, 18), (4, "fp32", 0.0, 60, 64), (5, "fp32", 0.0, 28, 30), (5, "fp32", 0.1, 20, 22),
    (6, "fp32_k64", 0.0, 12, 13), (8, "fp32_k64", 0.1, 4, 5), (9, "fp32_k64", 0.1, 4, 5)])
def test_where_stage_launches_are_faster(n1, precision, jitter, few, many):
    for k, resident in ((few, 1), (many, 0)):
        if k:
            m = _box(n1, (16, 16, k), jitter)
            s = _solver(m, precision)
            s.run(0.1 * m.computeMinNodeDistance(), 1)
            assert s.residentLaunches() == (resident, 0), k
            s.finalize()


def test_choices_for_stage_launches_leave_resident_launches_on():
    m = _box(5, (5, 4, 3))
    a = _solver(m, "fp32")
    a.run(1e-3, 2)
    a.tune()
    kept = a.segments()[0]
    a.finalize()
    # what a service applies in its next process
    b = _solver(m, "fp32")
    b.setSegmentOption(0, kept["option"], int(kept["stream_k"]))
    seg = b.segments()[0]
    assert (seg["option"], seg["stream_k"]) == (kept["option"], kept["stream_k"])
    b.run(1e-3, 2)
    b.setWalk(1)
    b.run(1e-3, 2)
    b.setWalk(-1)
    b.tune()
    b.run(1e-3, 2)
    assert b.residentLaunches() == (3, 0)
    b.finalize()


# what another process holds during a call by resident launches, by stage launches
@pytest.mark.parametrize("what,how", [("resident", fcntl.LOCK_EX), ("staged", fcntl.LOCK_SH)])
def test_another_process_steps_on_the_device(what, how):
    m = _box(6, (6, 5, 4))
    s = _solver(m, "fp32")
    s.run(1e-4, 3)
    held = [open(f) for f in glob.glob("/tmp/nekwave_amd.*.%s.lock" % what)]
    assert held
    for f in held:
        fcntl.flock(f, how | fcntl.LOCK_NB)  # free between calls
    s.run(1e-4, 2)
    assert s.residentLaunches() == (1, 0)
    for f in held:
        f.close()
    s.run(1e-4, 2)
    assert s.residentLaunches() == (2, 0)
    got = s.downloadState()
    s.finalize()
    r = _solver(m, "fp32", tile_option=0)
    r.run(1e-4, 7)
    assert np.array_equal(got, r.downloadState())
    r.finalize()


def test_solvers_of_one_device_share_it():
    # a solver that could run resident launches all the time, beside one of a mesh that cannot
    # (it gets a few stages in between two resident launches then: twenty times its time)
    a, b = _solver(_box(5, (8, 8, 8)), "fp32"), _solver(_box(8, (20, 20, 20)), "fp32")
    for s in (a, b):
        s.tune()
        s.run(1e-5, 20)

    def timed(n):
        t = []
        for _ in range(n):
            t0 = time.perf_counter()
            b.run(1e-5, 20)
            t.append(time.perf_counter() - t0)
        return float(np.median(t))

    alone = timed(9)
    stop = threading.Event()

    def keep_stepping():
        while not stop.is_set():
            a.run(1e-5, 100)

    th = threading.Thread(target=keep_stepping)
    th.start()
    try:
        time.sleep(0.05)
        beside = timed(9)
    finally:
        stop.set()
        th.join()
    assert a.residentLaunches()[1] == 0
    # an equal share of the GPU is twice the time alone, a launch in hand at the start some more
    assert beside < 6 * alone, (beside, alone)
    a.finalize()
    b.finalize()


def test_batches_of_several_launches():
    # (order, jitter, precision, cavities of k^3, resident launches per run): one launch; several
    # nearly full ones; too many for a jittered segment; places left empty; an order whose
    # segments run staged beyond one launch
    for n1, jitter, precision, k, count, launches in (
            (8, 0.0, "fp32", 6, 8, 1), (8, 0.0, "fp32", 8, 12, 3), (8, 0.1, "fp32", 8, 12, 3), (8, 0.1, "fp32", 8, 16, 0),
            (6, 0.0, "fp64", 11, 4, 0), (7, 0.0, "fp32", 12, 2, 2), (5, 0.0, "fp32", 12, 6, 0), (5, 0.0, "fp32", 8, 8, 1)):
        meshes = [_box(n1, (k, k, k), jitter) for _ in range(count)]
        b = nw.BatchSolver(precision=precision)
        b.initialize(meshes, 1.0)
        for x, m in enumerate(meshes):
            b.uploadState(x, np.ones(6 * m.getTotalPoints()))
        b.run(1e-3, 2)
        assert b.residentLaunches() == (launches, 0), (n1, jitter, precision, k)
        b.finalize()
    # the same order beside others, larger than the Infinity Cache together
    meshes = [_box(5, (8, 8, 8), 0.0) for _ in range(56)] + [_box(6, (12, 12, 12), 0.0) for _ in range(9)]
    b = nw.BatchSolver(precision="fp32")
    b.initialize(meshes, 1.0)
    for x, m in enumerate(meshes):
        b.uploadState(x, np.ones(6 * m.getTotalPoints()))
    b.run(1e-3, 1)
    assert b.residentLaunches() == (4 + 3, 0)
    b.finalize()


def test_a_launch_that_gives_up_is_counted(monkeypatch):
    m = _box(6, (10, 9, 8))
    s = _solver(m, "fp32")
    s.run(1e-4, 3)
    assert s.residentLaunches() == (1, 0)
    monkeypatch.setenv("NW_RESIDENT_SPINS", "0")  # the kernel's own bounded waits run out at once
    s.run(1e-4, 30)
    assert s.residentLaunches() == (1, 1)
    monkeypatch.delenv("NW_RESIDENT_SPINS")
    s.run(1e-4, 3)  # it keeps to stage launches
    assert s.residentLaunches() == (1, 1)
    got = s.downloadState()
    s.finalize()
    r = _solver(m, "fp32", tile_option=0)
    r.run(1e-4, 36)
    assert np.array_equal(got, r.downloadState())
    r.finalize()
