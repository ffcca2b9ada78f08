"""A frozen particle inside the lattice: its sites are left out of the iteration
vector, whose order the kernels take from a table made on the device. Residuals
against the oracle (sums of at most N = 19 terms of one sign and logarithms in
FP64: 1e-11 of the largest entry), products against finite differences of the
oracle's residual along the direction (central, h = 1e-5: h^2 and rounding / h,
1e-6)."""
import numpy as np
import pytest

from field_amd.spec import LatticeSpec, MoleculeSpec, SystemSpec

pytestmark = pytest.mark.gpu

CASES = {"1d": (LatticeSpec(1, (70,), lowerbound=("mirror1",), upperbound=("mirror1",)), [slice(20, 23)]),
         "2d": (LatticeSpec(2, (19, 57), lowerbound=("mirror1", "periodic"), upperbound=("mirror2", "periodic")),
                [slice(4, 7), slice(30, 60)]),
         "3d": (LatticeSpec(3, (9, 10, 17), lowerbound=("periodic",) * 3, upperbound=("periodic",) * 3),
                [slice(1, 4), slice(5, 6), slice(3, 9)])}


@pytest.mark.parametrize("name", CASES)
@pytest.mark.parametrize("chain", ["(A)19", "(A)7(B)8"])
def test_particle(sfx, orc, name, chain):
    lat, block = CASES[name]
    dims = lat.dims[: lat.gradients]
    wall = np.zeros(dims)
    wall[tuple(block)] = 1.0
    states = ("A", "B", "S", "W")
    chi = np.array([[0, 0.5, 0.4, -0.6], [0.5, 0, 0.3, 0.2], [0.4, 0.3, 0, 0], [-0.6, 0.2, 0, 0]])
    mols = [MoleculeSpec("p", chain, "restricted", theta=5.0), MoleculeSpec("b", "(B)3", "free", phibulk=0.02),
            MoleculeSpec("s", "(S)1", "solvent")]
    sysd = SystemSpec(states, chi, mols, frozen={"W": wall.reshape(-1)})
    G, O = sfx.System(lat, sysd), orc.System(lat, sysd)
    interior = wall[tuple(slice(1, n + 1) for n in lat.n_layers)]
    assert G.nvar == 3 * int((interior < 0.5).sum()) < 3 * interior.size
    rng = np.random.default_rng(6)
    x, v = rng.normal(0, 0.2, G.nvar), rng.normal(0, 1, G.nvar)
    f, fo = G.residual(x), O.residual(x)
    assert np.abs(f - fo).max() <= 1e-11 * np.abs(fo).max()
    d = (O.residual(x + 1e-5 * v) - O.residual(x - 1e-5 * v)) / 2e-5
    assert np.abs(G.jvp(x, v) - d).max() <= 1e-6 * np.abs(d).max()
