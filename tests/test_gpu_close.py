"""The launches that close an evaluation or a product (end sums, volume
fractions, contact averages, residuals) against the oracle: two to six states
(held in registers up to four), lattices of every kind, and site counts on both
sides of 65536, where the end sums take more threads.

Residual: sums of at most 8 products of one sign and 27 neighbours in another
order, 1e-12 of the largest entry. Product: the oracle's central difference with
step 1e-5, whose error is 1e-10 of third derivatives of order 10 and 1e-16 / 1e-5
of rounding: 1e-7 of the largest entry.
"""
import numpy as np
import pytest

from field_amd import sfx
from field_amd.spec import LatticeSpec, MoleculeSpec, SystemSpec

pytestmark = pytest.mark.gpu

LATTICES = {
    "flat_surface": LatticeSpec(2, (9, 7), lowerbound=("surface", "mirror1"), upperbound=("mirror2", "surface"), lambda_=0.2),
    "cylinder": LatticeSpec(2, (6, 11), geometry="cylindrical", lowerbound=("mirror1", "periodic"),
                            upperbound=("mirror1", "periodic"), lambda_=0.2),
    "sc": LatticeSpec(3, (6, 5, 7), lowerbound=("mirror1", "mirror2", "periodic"), upperbound=("mirror2", "mirror1", "periodic")),
    "fcc": LatticeSpec(3, (5, 6, 7), lattice_type="fcc", lowerbound=("periodic", "mirror1", "mirror2"),
                       upperbound=("periodic", "mirror1", "mirror1")),
    "hex": LatticeSpec(3, (4, 6, 5), lattice_type="hex", lowerbound=("periodic",) * 3, upperbound=("periodic",) * 3),
    "below_65536": LatticeSpec(2, (255, 256), lowerbound=("mirror1", "periodic"), upperbound=("mirror1", "periodic"), lambda_=0.2),
    "above_65536": LatticeSpec(2, (259, 256), lowerbound=("mirror1", "periodic"), upperbound=("mirror1", "periodic"), lambda_=0.2),
}


def system(lat, n_states):
    states = tuple("ABCDES"[:n_states - 1]) + ("S",)
    chi = np.zeros((n_states, n_states))
    for i in range(n_states):
        for j in range(i):
            chi[i, j] = chi[j, i] = 0.1 + 0.1 * ((i + 2 * j) % 5)
    mols = [MoleculeSpec("p", "".join(f"({s})2" for s in states[:-1]), "restricted", theta=0.2 * float(np.prod(lat.n_layers[:lat.gradients]))),
            MoleculeSpec("h", "(A)3", "free", phibulk=0.1), MoleculeSpec("s", "(S)1", "solvent")]
    return SystemSpec(states, chi, mols)


@pytest.mark.parametrize("name", LATTICES)
@pytest.mark.parametrize("n_states", [2, 3, 5, 6])
def test_close_matches_oracle(orc, name, n_states):
    print(name, n_states, flush=True)
    lat = LATTICES[name]
    sysd = system(lat, n_states)
    rng = np.random.default_rng(2)
    nv = sysd.nvar(lat)
    x, v = rng.normal(0, 0.1, nv), rng.normal(0, 1, nv)
    G, O = sfx.System(lat, sysd), orc.System(lat, sysd)
    f = O.residual(x)
    assert np.abs(G.residual(x) - f).max() <= 1e-12 * np.abs(f).max()
    d = (O.residual(x + 1e-5 * v) - O.residual(x - 1e-5 * v)) / 2e-5
    for _ in range(2):  # the ticket of the end sums is left at 0
        assert np.abs(G.jvp(x, v, precision="fp64") - d).max() <= 1e-7 * np.abs(d).max()
    G.compute_phi(x)
    O.compute_phi(x)
    for t in range(n_states):
        phi = O.phi(t)
        assert np.abs(G.phi(t) - phi).max() <= 1e-12 * np.abs(phi).max()
