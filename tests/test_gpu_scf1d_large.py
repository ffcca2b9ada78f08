"""One-workgroup evaluations of 1-D systems at the sizes where a lane holds two
and four layers (385 to 1024), on flat and curved lattices, with chains of two
state runs and of more than the 64 kept in registers, against the one-launch-
per-rank kernels: residuals are the same operations and the same bits; the
compiler fuses the last operations of a linearised residual in another order,
1e-14 of the largest entry."""
import numpy as np
import pytest

from test_gpu_scf1d import system

from field_amd import sfx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [385, 896, 897, 1024])
@pytest.mark.parametrize("geometry", ["flat", "cylindrical", "spherical"])
@pytest.mark.parametrize("chain", ["(A)9(B)8", "(A)1(B)1" * 40 + "(A)1", "(A)1(B)2" * 40 + "(A)3"],
                         ids=["two_runs", "palindrome_81_runs", "81_runs"])
def test_large_lattices(n, geometry, chain):
    print(n, geometry, flush=True)
    for bounds in (("surface", "mirror1"), ("mirror1", "surface")):
        lat, sysd = system(n, bounds, chain, geometry)
        rng = np.random.default_rng(8)
        A, B = sfx.System(lat, sysd), sfx.System(lat, sysd, sweep_kernel="per_rank")
        x, v = rng.normal(0, 0.1, A.nvar), rng.normal(0, 1, A.nvar)
        assert np.array_equal(A.residual(x), B.residual(x))
        a, b = A.jvp(x, v), B.jvp(x, v)
        assert np.abs(a - b).max() <= 1e-14 * np.abs(b).max()
