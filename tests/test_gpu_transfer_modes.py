"""downloadState and probeHistory where the caller's threads or memory are out of the
ordinary: threads that flush subnormals, and device memory for the arrays."""
import ctypes as C

import numpy as np
import pytest
import torch

import nekwave_amd as nw
from nekwave_amd import _lib

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


def test_arrays_in_device_memory():
    m = nw.Mesh(5)
    m.createBoxMesh(4, 3, 2, 0, 1, 0, 1, 0, 1, jitter=0.05, seed=1)
    n = 6 * m.getTotalPoints()
    st = np.random.default_rng(3).standard_normal(n)
    dp = C.POINTER(C.c_double)
    L = nw.lib()
    for precision, pipeline in (("fp64", "fused"), ("fp32", "fused"), ("fp64", "plain")):
        s = nw.DgSolver(precision=precision, pipeline=pipeline)
        s.initialize(m, 1.0)
        up, down = nw.DeviceBuffer.of(st), nw.DeviceBuffer(8 * n)
        _lib.check(L.nw_dg_upload(s._handle(), C.cast(up.ptr, dp), n))
        s.setProbes(m, [[0.3, 0.4, 0.5], [0.8, 0.1, 0.6]], capacity=4)
        s.sampleProbes()
        s.run(1e-3, 2)
        _lib.check(L.nw_dg_download(s._handle(), C.cast(down.ptr, dp), n))
        rec, nrec = nw.DeviceBuffer(8 * 4 * 2 * 6), C.c_int()
        _lib.check(L.nw_dg_probe_history(s._handle(), C.cast(rec.ptr, dp), 4, C.byref(nrec)))
        s.finalize()
        h = nw.DgSolver(precision=precision, pipeline=pipeline)
        h.initialize(m, 1.0)
        h.uploadState(st)
        h.setProbes(m, [[0.3, 0.4, 0.5], [0.8, 0.1, 0.6]], capacity=4)
        h.sampleProbes()
        h.run(1e-3, 2)
        assert np.array_equal(down.download(np.float64, n), h.downloadState())
        assert nrec.value == 3 and np.array_equal(rec.download(np.float64, 36).reshape(3, 2, 6), h.probeHistory())
        h.finalize()
