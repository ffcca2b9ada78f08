"""A 1-D system evaluated by one workgroup, and the batched problems, against
the one-launch-per-rank kernels, at lattice sizes around what a wave and a
workgroup hold (48, 384, 896 and 1024 layers), every bound, curved lattices,
and chains of one run, of a few and of more than the 64 kept in registers.

The single system repeats the per-rank kernels' operations, so the residual is
the same bits; its product too, up to the order in which the compiler fuses the
last operations of the linearised residual: 1e-14 of its largest entry. The
batch adds its sums in an order of its own: at most 1100 terms of one sign,
1e-12.
"""
import numpy as np
import pytest

from field_amd import configs, sfx
from field_amd.spec import LatticeSpec, MoleculeSpec, SystemSpec

pytestmark = pytest.mark.gpu

BOUNDS = [("surface", "mirror1"), ("mirror1", "surface"), ("mirror2", "mirror2"), ("periodic", "periodic"),
          ("mirror1", "mirror2")]
CHAINS = ["(A)2", "(A)3", "(A)17", "(A)9(B)8", "(A)16(B)33", "(A)1(B)1" * 40 + "(A)1", "(B)1(A)1" * 45]


def system(n, bounds, chain, geometry="flat"):
    lat = LatticeSpec(1, (n,), geometry=geometry, lowerbound=bounds[:1], upperbound=bounds[1:], lambda_=0.2,
                      offset_first_layer=2.0 if geometry != "flat" else 0.0)
    chi = np.array([[0.0, 0.7, 0.3, -0.8], [0.7, 0.0, 0.9, 0.0], [0.3, 0.9, 0.0, 0.0], [-0.8, 0.0, 0.0, 0.0]])
    wall = np.zeros(lat.M)
    frozen = {}
    if "surface" in bounds:
        wall[0 if bounds[0] == "surface" else n + 1] = 1.0
        frozen = {"W": wall}
    else:
        chi = chi[:3, :3]
    mols = [MoleculeSpec("p", chain, "restricted", theta=0.2 * n), MoleculeSpec("b", "(B)5", "free", phibulk=0.05),
            MoleculeSpec("s", "(S)1", "solvent")]
    return lat, SystemSpec(("A", "B", "S", "W")[: len(chi)], chi, mols, frozen=frozen)


def check(lat, sysd):
    rng = np.random.default_rng(8)
    A, B = sfx.System(lat, sysd), sfx.System(lat, sysd, sweep_kernel="per_rank")
    x, v = rng.normal(0, 0.1, A.nvar), rng.normal(0, 1, A.nvar)
    assert np.array_equal(A.residual(x), B.residual(x))
    for t in range(len(sysd.states)):
        assert np.array_equal(A.phi(t), B.phi(t))
    for m in range(len(sysd.molecules)):
        assert A.lngn(m) == B.lngn(m) and A.phibulk(m) == B.phibulk(m)
    assert A.free_energy() == B.free_energy()
    a, b = A.jvp(x, v), B.jvp(x, v)
    assert np.abs(a - b).max() <= 1e-14 * np.abs(b).max()


@pytest.mark.parametrize("n", [2, 8, 9, 10, 48, 49, 64, 65, 97, 384, 385, 897, 1024, 1025])
@pytest.mark.parametrize("bounds", BOUNDS)
def test_layers_and_bounds(n, bounds):
    print(n, bounds, flush=True)
    check(*system(n, bounds, "(A)9(B)8"))


@pytest.mark.parametrize("chain", CHAINS)
@pytest.mark.parametrize("geometry", ["flat", "cylindrical", "spherical"])
def test_chains_and_geometries(chain, geometry):
    print(geometry, chain[:20], flush=True)
    check(*system(57, ("surface", "mirror1"), chain, geometry))
    check(*system(57, ("mirror1", "surface"), chain, geometry))


@pytest.mark.parametrize("n_max", [8, 49, 97, 385, 449, 1024])
def test_batch_sizes(n_max):
    sizes = [n for n in (2, 3, 7, 8, 9, 47, 48, 49, 50, 96, 97, 192, 193, 384, 385, 448, 449, 1009, 1024) if n <= n_max]
    probs = [{"n_layers": n, "N": N, "chi_as": 0.4, "chi_s": -0.7, "phibulk": 0.02}
             for n in sizes for N in (2, 3, 4, 5, 17, 18, 19, 20, 33)]
    B = sfx.Batch(probs)
    x = np.random.default_rng(2).normal(0, 0.2, B.nvar)
    for p, f, xi in zip(probs, B.split(B.residual(x)), B.split(x)):
        lat, sysd, _ = configs.adsorption_problem(p)
        g = sfx.System(lat, sysd, sweep_kernel="per_rank").residual(xi)
        assert np.abs(f - g).max() <= 1e-12 * np.abs(g).max(), (p["n_layers"], p["N"])
