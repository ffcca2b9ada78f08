"""The several-ranks-per-launch kernel on FCC lattices against the
one-launch-per-rank kernels, at sides around its tile (8 x 8 x 16 sites, widened
by up to four) with every bound, and chain lengths that end in launches of one
to four ranks, palindromes and chains without a symmetry.

FP64: only the order of a site's twelve neighbours and of the composition's
terms differs, all of one sign, over at most N = 27 ranks: 1e-12 of the largest
entry. FP32: rounding of 1e-7 per rank: 2e-5.
"""
import numpy as np
import pytest

from field_amd import sfx
from field_amd.spec import LatticeSpec, MoleculeSpec, SystemSpec

pytestmark = pytest.mark.gpu

BOUNDS = [(("periodic",) * 3, ("periodic",) * 3),
          (("periodic", "mirror1", "mirror2"), ("periodic", "mirror1", "mirror1")),
          (("mirror2", "periodic", "mirror1"), ("mirror2", "periodic", "mirror2"))]


@pytest.mark.parametrize("sides", [(5, 5, 5), (8, 7, 16), (9, 17, 6), (12, 8, 33)])
@pytest.mark.parametrize("lo,hi", BOUNDS)
@pytest.mark.parametrize("palindrome", [True, False])
@pytest.mark.parametrize("n", [3, 7, 12])
def test_blocked_matches_per_rank(sides, lo, hi, palindrome, n):
    print(sides, lo, hi, palindrome, n, flush=True)
    lat = LatticeSpec(3, sides, lattice_type="fcc", lowerbound=lo, upperbound=hi)
    chi = np.array([[0.0, 0.7, 0.2], [0.7, 0.0, 0.9], [0.2, 0.9, 0.0]])
    chain = f"(A){n}(B)3(A){n}" if palindrome else f"(A){n}(B){n + 2}"
    sysd = SystemSpec(("A", "B", "S"), chi,
                      [MoleculeSpec("p", chain, "restricted", theta=0.2 * float(np.prod(sides))),
                       MoleculeSpec("s", "(S)1", "solvent")])
    rng = np.random.default_rng(4)
    nv = sysd.nvar(lat)
    x, v = rng.normal(0, 0.2, nv), rng.normal(0, 1, nv)
    B, P = sfx.System(lat, sysd), sfx.System(lat, sysd, sweep_kernel="per_rank")
    for precision, tol in (("fp64", 1e-12), ("fp32", 2e-5)):
        for what in ("residual", "jvp", "vjp"):
            arg = (x,) if what == "residual" else (x, v)
            a = getattr(B, what)(*arg, precision=precision)
            b = getattr(P, what)(*arg, precision=precision)
            assert np.abs(a - b).max() <= tol * np.abs(b).max(), (what, precision)
