"""Solvers driven from several threads: one thread's steps are captured into graphs while
others create solvers, change dt, transfer, probe and use the library's device buffers.
No call may fail for another's capture, and every state is that of a solver alone."""
import threading

import numpy as np
import pytest

import nekwave_amd as nw

pytestmark = pytest.mark.gpu


def _mesh(n1, nel):
    m = nw.Mesh(n1)
    m.createBoxMesh(*nel, 0, 1, 0, 1, 0, 1, True, False, False, jitter=0.1, seed=3)
    return m


def _round(m, precision, r, tile_option):
    s = nw.DgSolver(precision=precision, tile_option=tile_option)
    s.initialize(m, 1.0)
    s.uploadState(np.random.default_rng(r).standard_normal(6 * m.getTotalPoints()))
    s.setProbes(m, [[0.3, 0.4, 0.5]], capacity=8)
    for k in range(3):
        s.run(1e-4 * (1 + k + r % 3), 2)  # another dt each time; both graphs of the step
    out = [s.downloadState(), s.probeHistory(), np.array(list(s.diagnostics().values()))]
    b = nw.DeviceBuffer.of(out[0])
    out.append(b.download(np.float64, out[0].size))
    b.free()
    s.finalize()
    return out


def test_captures_beside_other_threads_calls():
    jobs = [(_mesh(4, (3, 2, 2)), "fp64", 0), (_mesh(5, (2, 2, 3)), "fp32", 0), (_mesh(6, (2, 2, 2)), "fp32", -1),
            (_mesh(3, (4, 3, 3)), "fp64", -1)]
    want = [[_round(m, p, r, o) for r in range(3)] for m, p, o in jobs]
    failed = []
    start = threading.Barrier(len(jobs))

    def go(x):
        m, p, o = jobs[x]
        start.wait()
        try:
            for r in range(30):
                got = _round(m, p, r % 3, o)
                if not all(np.array_equal(a, b) for a, b in zip(got, want[x][r % 3])):
                    failed.append((x, r))
        except nw.NekWaveError as e:
            failed.append((x, str(e)))

    ts = [threading.Thread(target=go, args=(x,)) for x in range(len(jobs))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not failed
