"""downloadState and probeHistory where the caller's threads or memory are out of the
ordinary: threads that flush subnormals, and device memory for the arrays."""
import numpy as np
import pytest
import torch

import nekwave_amd as nw

pytestmark = pytest.mark.gpu


# one worker; several workers and chunks
@pytest.mark.parametrize("n1,nel", [(4, (3, 3, 3)), (8, (12, 11, 11))])
def test_download_keeps_subnormals_where_threads_flush_them(n1, nel):
    m = nw.Mesh(n1)
    m.createBoxMesh(*nel, 0, 1, 0, 1, 0, 1)
    n = 6 * m.getTotalPoints()
    # FP32's subnormal range, and values around its edges
    st = np.random.default_rng(1).standard_normal(n) * 10.0 ** np.random.default_rng(2).uniform(-45, -36, n)
    want = st.astype(np.float32).astype(np.float64).view(np.int64)
    s = nw.DgSolver(precision="fp32")
    s.initialize(m, 1.0)
    s.uploadState(st)
    assert torch.set_flush_denormal(True)
    try:
        got = s.downloadState()
    finally:
        torch.set_flush_denormal(False)
    s.finalize()
    assert np.array_equal(got.view(np.int64), want)
