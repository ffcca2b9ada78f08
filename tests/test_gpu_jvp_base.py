"""A Jacobian product sweeps base and tangent propagators together; the base
results it leaves (phi, ln G_N, bulk fractions) are those of compute_phi at the
same x, on every system of the parity set.

FP64: the same terms, composed in another order (at most 24 of them): 1e-13 of
the largest. FP32: both carry rounding of 1e-7 per rank over at most 24 ranks
and two chains, 1e-5.
"""
import numpy as np
import pytest

import cases
from field_amd import sfx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", cases.NAMES)
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-13), ("fp32", 1e-5)])
def test_jvp_leaves_the_base_of_compute_phi(name, precision, tol):
    lat, sysd = cases.case(name)
    x = cases.start(lat, sysd)
    v = np.random.default_rng(3).normal(0, 1, x.size)
    A, B = sfx.System(lat, sysd), sfx.System(lat, sysd)
    A.jvp(x, v, precision=precision)
    B.compute_phi(x, precision=precision)
    for t in range(len(sysd.states)):
        a, b = A.phi(t), B.phi(t)
        assert np.abs(a - b).max() <= tol * max(np.abs(b).max(), 1e-300)
    for m in range(len(sysd.molecules)):
        assert abs(A.lngn(m) - B.lngn(m)) <= tol * max(1.0, abs(B.lngn(m)))
        assert abs(A.phibulk(m) - B.phibulk(m)) <= tol * max(1.0, abs(B.phibulk(m)))
