"""The kernel-level launchers whose kernels are compiled per n1 (volume curl, lift) or
place their blocks by chiplet (restrict, flux), at every n1 and at element counts that
leave workgroups and the last block incomplete, against the oracle.

Tolerances: volume 1e-13 of the largest value (3 n1 products per derivative, eps 1e-16
each), lift and flux 1e-14 (at most about 20 roundings), restrict bit-exact.
"""
import numpy as np
import pytest

import pyoracle as po
from nekwave_amd import DeviceBuffer as DB
from nekwave_amd._lib import check, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nel", [(1, 1, 1), (5, 3, 1)])
@pytest.mark.parametrize("n1", range(2, 11))
def test_against_oracle(n1, nel):
    o = po.Mesh.box(n1, nel, (0, 1.5, 0, 1, 0, 1), (1, 0, 0), jitter=0.05, seed=4)
    rng = np.random.default_rng(n1)
    S, T = o.npts, o.tfp
    st = rng.standard_normal(6 * S)
    ref = po.volume_curl(o, st[:S], st[S:2 * S], st[2 * S:3 * S], -1.0)
    d_st, dw = DB.of(st), DB(8 * 3 * S)
    b = {k: DB.of(getattr(o, k)) for k in ("D", "w3", "jac", "rx", "sx", "tx", "ry", "sy", "ty", "rz", "sz", "tz")}
    check(lib().nw_launch_volume_curl(*(d_st.offset(8 * S * c) for c in range(3)), *(dw.offset(8 * S * c) for c in range(3)),
                                      *(x.ptr for x in b.values()), -1.0, n1, o.nelt, None))
    fEN, fHN = po.restrict(o, st, S)
    d = {k: DB.of(getattr(o, k)) for k in ("vM", "vP", "bc", "nx", "ny", "nz", "dA")}
    d_fE, d_fH, d_fl = DB(8 * 3 * T), DB(8 * 3 * T), DB(8 * 6 * T)
    check(lib().nw_launch_restrict_faces(d_st.ptr, d_fE.ptr, d_fH.ptr, d["vM"].ptr, T, S, None))
    check(lib().nw_launch_compute_flux(d_st.ptr, d_fE.ptr, d_fH.ptr, d["vP"].ptr, d["bc"].ptr, d["nx"].ptr, d["ny"].ptr,
                                       d["nz"].ptr, d_fl.ptr, 1.0, T, S, d["vM"].ptr, None, None, None, o.np, S, None))
    rhs0 = rng.standard_normal(6 * S)
    d_rhs = DB.of(rhs0)
    check(lib().nw_dev_sync())
    fl = po.flux(o, st, fEN, fHN, 1.0, S)
    got = dw.download(np.float64, 3 * S)
    for c in range(3):
        np.testing.assert_allclose(got[c * S:(c + 1) * S], ref[c], rtol=0, atol=1e-13 * np.abs(ref[c]).max())
    assert np.array_equal(d_fE.download(np.float64, 3 * T), fEN)
    assert np.array_equal(d_fH.download(np.float64, 3 * T), fHN)
    np.testing.assert_allclose(d_fl.download(np.float64, 6 * T), fl, rtol=0, atol=1e-14 * np.abs(fl).max())
    d_fl.upload(fl)  # the lift on its own
    check(lib().nw_launch_add_flux(d_fl.ptr, d["vM"].ptr, d["dA"].ptr, d_rhs.ptr, T, S, None))
    check(lib().nw_dev_sync())
    rhs = po.add_flux(o, fl, rhs0)
    np.testing.assert_allclose(d_rhs.download(np.float64, 6 * S), rhs, rtol=0, atol=1e-14 * np.abs(rhs).max())
