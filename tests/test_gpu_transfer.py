"""uploadState and downloadState at the sizes where their route changes (staging
slots, the runtime's copy, one or several chunks and workers): what comes back is
what went up -- bit for bit in FP64, rounded to FP32 once in FP32 -- and several
threads' transfers do not mix."""
import threading

import numpy as np
import pytest

import nekwave_amd as nw

pytestmark = pytest.mark.gpu


def _mesh(n1, nel):
    m = nw.Mesh(n1)
    m.createBoxMesh(*nel, 0, 1, 0, 1, 0, 1)
    return m


# nodes: 8; 21952 (just over 1 MB); 87808 (4 MB); 699392 (33.6 MB: several chunks, ragged last one)
@pytest.mark.parametrize("n1,nel", [(2, (1, 1, 1)), (7, (4, 4, 4)), (7, (8, 8, 4)), (8, (11, 11, 11)), (8, (12, 11, 11))])
@pytest.mark.parametrize("precision,pipeline", [("fp64", "fused"), ("fp32", "fused"), ("fp64", "plain")])
def test_round_trip(n1, nel, precision, pipeline):
    m = _mesh(n1, nel)
    st = np.random.default_rng(1).standard_normal(6 * m.getTotalPoints()) * 10.0 ** np.random.default_rng(2).uniform(
        -44, 30, 6 * m.getTotalPoints())  # FP32's subnormal range among them
    st[:3] = [0.0, -0.0, 1e-300]
    s = nw.DgSolver(precision=precision, pipeline=pipeline)
    s.initialize(m, 1.0)
    want = st if precision == "fp64" else st.astype(np.float32).astype(np.float64)
    for _ in range(2):
        s.uploadState(st)
        assert np.array_equal(s.downloadState(), want)
    s.finalize()


def test_transfers_from_several_threads():
    sizes = [(8, (9, 9, 9)), (6, (5, 5, 5)), (8, (12, 11, 11)), (5, (3, 3, 3))]
    bad = []

    def one(x, n1, nel):
        m = _mesh(n1, nel)
        s = nw.DgSolver(precision="fp32" if x % 2 else "fp64")
        s.initialize(m, 1.0)
        for r in range(4):
            st = np.random.default_rng(10 * x + r).standard_normal(6 * m.getTotalPoints())
            s.uploadState(st)
            if not np.array_equal(s.downloadState(), st if x % 2 == 0 else st.astype(np.float32).astype(np.float64)):
                bad.append((x, r))
        s.finalize()

    ts = [threading.Thread(target=one, args=(x, *c)) for x, c in enumerate(sizes)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
