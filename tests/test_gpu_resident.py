"""The resident multi-step launch (meshes that fit on chip; any number of steps
per launch, traces exchanged as tagged packets) against the stage launches of an
explicit tile option: the same expressions in the same order, so the same bits --
at every n1 and precision, from one element to several elements per workgroup,
in batches cut into several launches, with probes, and where a launch gives up
waiting and its steps are run again by stage launches."""
import numpy as np
import pytest

import nekwave_amd as nw

pytestmark = pytest.mark.gpu


def _mesh(n1, nel, per=(True, False, False), jitter=0.1, media=True, seed=3):
    m = nw.Mesh(n1)
    m.createBoxMesh(*nel, 0, 1, 0, 1, 0, 1, *per, jitter=jitter, seed=seed)
    if media:
        rng = np.random.default_rng(seed)
        n = nel[0] * nel[1] * nel[2]
        m.setMaterials(rng.uniform(1, 4, n), rng.uniform(0.5, 2, n))
    return m


def _both(m, precision, nsteps, groups_per_cu=0, runs=2):
    st0 = np.random.default_rng(7).standard_normal(6 * m.getTotalPoints())
    dt = 0.4 * m.computeMinNodeDistance()
    out = []
    for opt in (-1, 0):
        s = nw.DgSolver(precision=precision, tile_option=opt, groups_per_cu=groups_per_cu)
        s.initialize(m, 1.0)
        s.uploadState(st0)
        for _ in range(runs):
            s.run(dt, nsteps)
        out.append(s.downloadState())
        s.finalize()
    return out


@pytest.mark.parametrize("precision", ["fp64", "fp32", "fp32_k64"])
@pytest.mark.parametrize("n1", range(2, 10))
def test_resident_steps_equal_stage_launches(n1, precision):
    # one element (its own periodic neighbour), a ragged box, uniform and jittered;
    # with one workgroup per CU the last two need several elements per workgroup
    for nel, kw, cap in (((1, 1, 1), {"jitter": 0.0, "per": (True, True, True)}, 0), ((3, 2, 5), {}, 0),
                         ((5, 4, 3), {"jitter": 0.0, "media": False}, 0), ((9, 7, 5), {}, 1),
                         ((13, 9, 5), {"jitter": 0.0}, 1)):
        a, b = _both(_mesh(n1, nel, **kw), precision, 3, cap)
        assert np.array_equal(a, b), (nel, np.abs(a - b).max())


@pytest.mark.parametrize("n1,nel", [(8, (11, 11, 11)), (7, (16, 16, 8)), (5, (20, 16, 16)), (9, (12, 12, 12)), (6, (12, 13, 14)), (4, (17, 17, 17))])
def test_resident_up_to_the_chip(n1, nel):
    a, b = _both(_mesh(n1, nel), "fp32", 2, runs=1)
    assert np.array_equal(a, b)


def test_resident_batch_in_several_launches():
    # one workgroup per CU: the n1 = 5 cavities fill more than one launch
    meshes = [_mesh(n1, (k, k, k), (False,) * 3, 0.0, seed=x)
              for x, (n1, k) in enumerate([(5, 10), (4, 3), (5, 9), (5, 2), (7, 4), (5, 10), (4, 2)])]
    ics = [np.random.default_rng(x).standard_normal(6 * m.getTotalPoints()) for x, m in enumerate(meshes)]
    got = []
    for opt in (-1, 0):
        s = nw.BatchSolver(precision="fp32", tile_option=opt, groups_per_cu=1)
        s.initialize(meshes, 1.0)
        for x, u in enumerate(ics):
            s.uploadState(x, u)
        s.run(1e-3, 4)
        s.run(1e-3, 1)
        got.append([s.downloadState(x) for x in range(len(meshes))])
        s.finalize()
    for a, b in zip(*got):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("spins", [None, "0"])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_resident_probes_and_a_launch_that_gives_up(precision, spins, monkeypatch):
    if spins is not None:  # the kernel's own bounded waits run out at once; every launch still ends
        monkeypatch.setenv("NW_RESIDENT_SPINS", spins)
    m = _mesh(6, (7, 6, 5))
    pts = np.random.default_rng(5).uniform(0.05, 0.95, (5, 3))
    pts[3] = pts[1] + 1e-4  # two probes in one element
    st0 = np.random.default_rng(7).standard_normal(6 * m.getTotalPoints())
    got = []
    for opt in (-1, 0):
        s = nw.DgSolver(precision=precision, tile_option=opt)
        s.initialize(m, 1.0)
        s.uploadState(st0)
        s.setProbes(m, pts, capacity=16)
        s.sampleProbes()
        rec = []
        for n in (1, 7, 8):
            s.run(1e-3, n)
            rec.append(s.probeHistory())
        got.append((s.downloadState(), np.concatenate(rec), s.diagnostics()))
        s.finalize()
    assert got[0][1].shape == (17, 5, 6)
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1]) and got[0][2] == got[1][2]
