"""Timings where a resident launch gives up waiting: time() measures the stage launches
the solver then keeps to, and the state, the probe records and the steps after it are
those of a solver that ran stage launches from the start."""
import numpy as np
import pytest

import nekwave_amd as nw

pytestmark = pytest.mark.gpu

WARMUP, STEPS, REPEATS = 3, 40, 4


@pytest.mark.parametrize("probes", [False, True])
def test_times_cover_the_steps_after_a_launch_gave_up(probes, monkeypatch):
    monkeypatch.setenv("NW_RESIDENT_SPINS", "0")  # the kernel's own bounded waits run out at once
    m = nw.Mesh(6)
    m.createBoxMesh(10, 9, 8, 0, 1, 0, 1, 0, 1, True, False, False, jitter=0.1, seed=3)
    st0 = np.random.default_rng(7).standard_normal(6 * m.getTotalPoints())
    dt = 0.2 * m.computeMinNodeDistance()
    got, ms = [], []
    for opt in (-1, 0):
        s = nw.DgSolver(precision="fp32", tile_option=opt)
        s.initialize(m, 1.0)
        s.uploadState(st0)
        if probes:
            s.setProbes(m, [[0.3, 0.4, 0.5], [0.7, 0.2, 0.9]], capacity=256)
        ms.append(s.timeRepeats(dt, STEPS, REPEATS, warmup=WARMUP))
        end = s.downloadState()
        rec = s.probeHistory() if probes else np.zeros(0)
        s.run(dt, 5)
        got.append((end, rec, s.downloadState(), s.probeHistory() if probes else np.zeros(0)))
        s.finalize()
    if probes:
        assert got[0][1].shape == (WARMUP + REPEATS * STEPS, 2, 6) and got[0][3].shape[0] == 5
    for a, b in zip(*got):
        assert np.array_equal(a, b)
    # the same work on stage launches; a tuned shape is at most a few times faster than
    # option 0, an abandoned launch takes microseconds
    assert ms[0].min() > 0.25 * ms[1].min(), ms
