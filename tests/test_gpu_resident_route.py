"""Which launches run: a mesh that fits on chip takes resident launches and every one of
them completes, from one workgroup per CU up to the largest mesh the launcher places
(an overestimate would show as launches that give up, whose steps run again by stage
launches with the same result), and one that gives up is counted as such."""
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
            assert done == 1 or (done == 0 and k > 1), (jitter, k)
            if done == 0:  # does not fit
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
