"""The several-ranks-per-launch kernel of 2-D lattices against the one-launch-
per-rank kernels, at sides around its tile (8 x 48 sites, widened by eight) and
smaller than its widening, with every bound, flat and cylindrical, and chain
lengths that end in launches of one to eight ranks.

The two run the same recursion. In FP64 only the order in which a site's
composition and a mirrored neighbour's terms are summed differs, at most N
terms of one sign: 1e-12 of the largest entry. In FP32 both carry rounding of
1e-7 per rank over at most 43 ranks.
"""
import numpy as np
import pytest

from field_amd import sfx
from field_amd.spec import LatticeSpec, MoleculeSpec, SystemSpec

pytestmark = pytest.mark.gpu

SIDES = [(2, 2), (3, 48), (8, 7), (9, 49), (16, 97), (25, 56), (41, 17)]
FLAT = [(("mirror1", "mirror2"), ("mirror2", "mirror1")), (("periodic", "surface"), ("periodic", "mirror1")),
        (("surface", "periodic"), ("surface", "periodic"))]
CURVED = [(("mirror1", "mirror1"), ("surface", "mirror1")), (("mirror1", "periodic"), ("mirror1", "periodic"))]


def system(sides, lo, hi, geometry, n):
    lat = LatticeSpec(2, sides, geometry=geometry, lowerbound=lo, upperbound=hi, lambda_=0.2)
    chi = np.array([[0.0, 0.8, 0.4], [0.8, 0.0, 0.6], [0.4, 0.6, 0.0]])
    mols = [MoleculeSpec("p", f"(A){n}(B){n + 3}", "restricted", theta=0.3 * float(np.prod(sides))),
            MoleculeSpec("h", f"(B){2 * n + 1}", "free", phibulk=0.1), MoleculeSpec("s", "(S)1", "solvent")]
    return lat, SystemSpec(("A", "B", "S"), chi, mols)


@pytest.mark.parametrize("sides", SIDES)
@pytest.mark.parametrize("geometry,lo,hi", [("flat", *b) for b in FLAT] + [("cylindrical", *b) for b in CURVED])
@pytest.mark.parametrize("n", [2, 9, 20])
def test_blocked_matches_per_rank(sides, geometry, lo, hi, n):
    print(sides, geometry, lo, hi, n, flush=True)
    lat, sysd = system(sides, lo, hi, geometry, n)
    rng = np.random.default_rng(4)
    nv = sysd.nvar(lat)
    x, v = rng.normal(0, 0.2, nv), rng.normal(0, 1, nv)
    B, P = sfx.System(lat, sysd), sfx.System(lat, sysd, sweep_kernel="per_rank")
    for precision, tol in (("fp64", 1e-12), ("fp32", 2e-5)):
        if precision == "fp32" and P.phibulk(2) < 0:
            continue  # a slit's chains leave the solvent a negative bulk: phi_total cancels, which FP32 cannot hold
        for what in ("residual", "jvp", "vjp"):
            arg = (x,) if what == "residual" else (x, v)
            a = getattr(B, what)(*arg, precision=precision)
            b = getattr(P, what)(*arg, precision=precision)
            assert np.abs(a - b).max() <= tol * np.abs(b).max(), (what, precision)
