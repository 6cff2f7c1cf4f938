"""The plain pipeline's stage kernel (one launch per stage) against the FP64 oracle over
every n1 it takes, at element counts around its workgroups (one element, a workgroup
with missing elements, a grid that is no multiple of the eight chiplets), with walls,
periodic faces, media and the halo stand-in.

Tolerance: 1e-12 relative L2, the FP64 bound of test_gpu_solver.py (10 stages of
rounding differences of order 1e-15 each, amplified by at most the derivative
matrix's norm times dt).
"""
import numpy as np
import pytest

from gpu_util import pair, random_state, rel_l2, run_oracle, run_product

pytestmark = pytest.mark.gpu

# (nel, periodic, media, halo)
SHAPES = [((1, 1, 1), (0, 0, 0), False, False),
          ((17, 1, 1), (0, 0, 0), True, False),
          ((3, 3, 2), (1, 0, 1), True, True)]


@pytest.mark.parametrize("shape", range(len(SHAPES)))
@pytest.mark.parametrize("n1", range(2, 11))
def test_matches_oracle(n1, shape):
    nel, per, media, halo = SHAPES[shape]
    nelt = nel[0] * nel[1] * nel[2]
    eps = mu = None
    if media:
        rng = np.random.default_rng(n1)
        eps, mu = np.exp(0.3 * rng.standard_normal(nelt)), np.exp(0.3 * rng.standard_normal(nelt))
    m, o = pair(n1, nel, (0, 1, 0, 1, 0, 1), per, 0.0 if halo else 0.05, 3, eps, mu, halo)
    st0 = random_state(o, n1)
    dt = 0.5 * o.auto_dt()
    ref = run_oracle(o, st0, dt, 2, 1.0)
    got = run_product(m, st0, dt, 2, 1.0, "fp64", "plain")
    err = rel_l2(o, got, ref)
    print("n1=%d %s relL2=%.3e" % (n1, nel, err))
    assert err <= 1e-12, err
