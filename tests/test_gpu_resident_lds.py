"""Resident launches whose workgroups keep LSRK registers of some or all of their
elements in LDS (many elements per workgroup, per-node geometry, FP64 registers),
against the stage launches of an explicit tile option: the same bits."""
import numpy as np
import pytest

import nekwave_amd as nw

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,n1,nel", [
    ("fp64", 2, (12, 12, 13)), ("fp64", 3, (14, 14, 14)), ("fp64", 4, (14, 14, 13)), ("fp64", 5, (10, 10, 10)),
    ("fp32", 5, (16, 16, 16)), ("fp32", 4, (20, 19, 17)), ("fp32_k64", 5, (16, 16, 15)), ("fp32_k64", 7, (13, 9, 11)),
    ("fp32_k64", 8, (10, 10, 9))])
def test_same_bits_as_stage_launches(precision, n1, nel):
    m = nw.Mesh(n1)
    m.createBoxMesh(*nel, 0, 1, 0, 1, 0, 1, True, False, False, jitter=0.1, seed=3)
    st0 = np.random.default_rng(7).standard_normal(6 * m.getTotalPoints())
    dt = 0.4 * m.computeMinNodeDistance()
    out = []
    for opt in (-1, 0):
        s = nw.DgSolver(precision=precision, tile_option=opt)
        s.initialize(m, 1.0)
        s.uploadState(st0)
        s.run(dt, 2)
        s.run(dt, 1)
        out.append(s.downloadState())
        s.finalize()
    assert np.array_equal(*out)
