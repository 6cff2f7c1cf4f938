"""Resident launches where one call takes several of them (long runs, many probed
elements), where a later one gives up, beside staged segments of the same batch, beside
another thread's solver, and on meshes whose elements have rotated frames: the bits of
stage launches, on the route that the test is about."""
import threading

import numpy as np
import pytest

import nekwave_amd as nw
import test_meshio as meshio
from gpu_util import rel_l2, run_oracle

pytestmark = pytest.mark.gpu


def _box(n1, nel, jitter=0.1, seed=3):
    m = nw.Mesh(n1)
    m.createBoxMesh(*nel, 0, 1, 0, 1, 0, 1, True, False, False, jitter=jitter, seed=seed)
    return m


def _state(m, seed=7):
    return np.random.default_rng(seed).standard_normal(6 * m.getTotalPoints())


def _solver(m, precision, **kw):
    s = nw.DgSolver(precision=precision, **kw)
    s.initialize(m, 1.0)
    s.uploadState(_state(m))
    return s


# a launch takes about 10 ms of steps, here 777, and a call waits after three of them
@pytest.mark.parametrize("spins,launches", [(None, (4, 0)), ("1000000,0", (1, 1)), ("1000000,1000000,0", (2, 1))])
def test_a_long_run_in_several_launches(spins, launches, monkeypatch):
    m = _box(3, (5, 4, 3))
    dt = 0.2 * m.computeMinNodeDistance()
    ref = _solver(m, "fp64", tile_option=0)
    ref.run(dt, 2500)
    want = ref.downloadState()
    ref.finalize()
    if spins is not None:  # from the second or third launch on, the waits run out at once
        monkeypatch.setenv("NW_RESIDENT_SPINS", spins)
    s = _solver(m, "fp64")
    s.run(dt, 2500)
    assert s.residentLaunches() == launches
    assert np.isfinite(want).all() and np.array_equal(s.downloadState(), want)
    s.finalize()


@pytest.mark.parametrize("spins,complete", [(None, True), ("1000000,0", False)])
def test_more_steps_than_a_launch_keeps_for_the_probes(spins, complete, monkeypatch):
    # 150 probed elements of n1 = 9 in FP64 are 5.2 MB a step: a launch keeps six steps
    m = _box(9, (6, 5, 5))
    pts = (np.stack(np.meshgrid(np.arange(6) + 0.5, np.arange(5) + 0.5, np.arange(5) + 0.5), -1).reshape(-1, 3)
           / np.array([6, 5, 5]))
    dt = 0.2 * m.computeMinNodeDistance()
    got = []
    for opt in (0, -1):
        if opt == -1 and spins is not None:
            monkeypatch.setenv("NW_RESIDENT_SPINS", spins)
        s = _solver(m, "fp64", tile_option=opt)
        s.setProbes(m, pts, capacity=40)
        s.run(dt, 20)
        rec = s.probeHistory()
        assert rec.shape == (20, 150, 6)
        if opt == -1:
            done, lost = s.residentLaunches()
            assert (done >= 4 and lost == 0) if complete else (done, lost) == (1, 1)
        got.append((rec, s.downloadState()))
        s.finalize()
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])


def test_batch_with_staged_and_resident_segments():
    # the n1 = 7 segment is too large for the chip; the others fit.  After an odd number of steps
    # in one call and a call that finds the place taken, the segments' buffers differ
    meshes = [_box(5, (4, 3, 2)), _box(7, (16, 16, 12), 0.05), _box(4, (5, 4, 3), 0.0), _box(5, (2, 3, 4), seed=9)]
    ics = [_state(m, x) for x, m in enumerate(meshes)]
    got = []
    for opt in (0, -1):
        b = nw.BatchSolver(precision="fp32", tile_option=opt)
        b.initialize(meshes, 1.0)
        for x, u in enumerate(ics):
            b.uploadState(x, u)
        for n in (1, 3, 1030, 2):
            b.run(1e-5, n)
        b.uploadState(2, ics[2])
        b.run(1e-5, 1)
        if opt == -1:
            assert b.residentLaunches() == (2 * 6, 0)  # two segments; 1030 steps are two launches each
        got.append([b.downloadState(x) for x in range(len(meshes))] + [np.array(list(b.diagnostics(x).values())) for x in range(4)])
        b.finalize()
    for a, c in zip(*got):
        assert np.array_equal(a, c)


def test_two_solvers_of_one_device_in_two_threads():
    m = [_box(5, (5, 4, 3)), _box(6, (4, 4, 3), 0.0)]
    dt = [0.2 * x.computeMinNodeDistance() for x in m]
    want = []
    for x in range(2):
        r = _solver(m[x], "fp32", tile_option=0)
        r.run(dt[x], 600)
        want.append(r.downloadState())
        r.finalize()
    s = [_solver(x, "fp32") for x in m]
    for x in s:
        x.tune()
    start = threading.Barrier(2)

    def go(x):
        start.wait()
        for _ in range(60):
            s[x].run(dt[x], 10)

    ts = [threading.Thread(target=go, args=(x,)) for x in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for x in range(2):
        done, lost = s[x].residentLaunches()
        assert lost == 0 and done <= 60  # calls that found the place taken ran by stage launches
        assert np.array_equal(s[x].downloadState(), want[x])
        s[x].finalize()


# n1 = 8: the quad-broadcast volume; the last: several elements per workgroup
@pytest.mark.parametrize("n1,nel,cap", [(4, (3, 3, 3), 0), (5, (3, 4, 3), 0), (8, (3, 3, 2), 0), (7, (3, 3, 3), 0), (4, (7, 7, 6), 1)])
def test_rotated_element_frames(n1, nel, cap):
    corners = meshio.block_mesh(nel, meshio.rotations(), h=0.5, skew=0.1, seed=n1)
    ne, nf = meshio.adjacency(corners)
    kind = np.where(ne >= 0, nw.FACE_E, nw.FACE_PEC).astype(np.int32)
    m = nw.Mesh.fromCorners(n1, corners, kind.reshape(-1, 6), ne.reshape(-1, 6).astype(np.int32), nf.reshape(-1, 6).astype(np.int32))
    o = meshio.product_to_oracle(m)
    st0 = _state(m)
    dt = 0.3 * o.auto_dt()
    ref = run_oracle(o, st0, dt, 5)
    for precision, tol in (("fp64", 1e-12), ("fp32", 2e-5), ("fp32_k64", 2e-5)):
        got = []
        for opt in (-1, 0):
            s = nw.DgSolver(precision=precision, tile_option=opt, groups_per_cu=cap)
            s.initialize(m, 1.0)
            s.uploadState(st0)
            s.run(dt, 5)
            got.append(s.downloadState())
            assert s.residentLaunches() == ((1, 0) if opt == -1 else (0, 0))
            s.finalize()
        assert np.array_equal(*got)
        assert rel_l2(o, got[0], ref) <= tol
