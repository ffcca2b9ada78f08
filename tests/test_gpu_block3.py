"""The several-ranks-per-launch kernel of the 3-D simple-cubic lattice against
the one-launch-per-rank kernels, at sides around its tile (8 x 8 x 16 sites,
widened by up to four) and chain lengths that end in launches of one to four
ranks.

The two run the same recursion. In FP64 only the order in which a site's
composition is summed differs: at most N terms, so N ulps of phi, and less than
1e-12 of the residual's and the product's largest entry for these chains. In
FP32 both carry rounding of 1e-7 per rank over at most 23 ranks.
"""
import numpy as np
import pytest

from field_amd import sfx
from field_amd.spec import LatticeSpec, MoleculeSpec, SystemSpec

pytestmark = pytest.mark.gpu

SIDES = [(5, 5, 5), (8, 8, 16), (9, 7, 17), (7, 16, 15), (16, 9, 33), (6, 25, 31)]
LO, HI = ("mirror1", "mirror2", "periodic"), ("mirror2", "mirror1", "periodic")


def system(sides, n):
    lat = LatticeSpec(3, sides, lowerbound=LO, upperbound=HI)
    chi = np.array([[0.0, 0.8, 0.4], [0.8, 0.0, 0.6], [0.4, 0.6, 0.0]])
    v = float(np.prod(sides))
    mols = [MoleculeSpec("p", f"(A){n}(B){n + 2}", "restricted", theta=0.3 * v),
            MoleculeSpec("h", f"(B){2 * n + 1}", "free", phibulk=0.1), MoleculeSpec("s", "(S)1", "solvent")]
    return lat, SystemSpec(("A", "B", "S"), chi, mols)


@pytest.mark.parametrize("sides", SIDES)
@pytest.mark.parametrize("n", [2, 5, 10])
@pytest.mark.parametrize("schedule", ["auto", "sequential"])
def test_blocked_matches_per_rank(sides, n, schedule):
    lat, sysd = system(sides, n)
    rng = np.random.default_rng(4)
    nv = sysd.nvar(lat)
    x, v = rng.normal(0, 0.2, nv), rng.normal(0, 1, nv)
    B = sfx.System(lat, sysd, sweep_kernel="blocked", chain_schedule=schedule)
    P = sfx.System(lat, sysd, sweep_kernel="per_rank")
    for precision, tol in (("fp64", 1e-12), ("fp32", 2e-5)):
        for what in ("residual", "jvp", "vjp"):
            arg = (x,) if what == "residual" else (x, v)
            a = getattr(B, what)(*arg, precision=precision)
            b = getattr(P, what)(*arg, precision=precision)
            assert np.abs(a - b).max() <= tol * np.abs(b).max(), (what, precision)
