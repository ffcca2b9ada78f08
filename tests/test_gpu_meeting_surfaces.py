"""2-D lattices whose surfaces meet in a corner: the contact average there takes the
two neighbours on the lattice, and enters the free energy and the grand potential.
Against the oracle: sums over at most 1300 sites of terms of both signs, 1e-11 of
the value or of 1."""
import itertools

import numpy as np
import pytest

from field_amd.spec import LatticeSpec, MoleculeSpec, SystemSpec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sides", [(2, 2), (3, 9), (21, 58)])
@pytest.mark.parametrize("geometry", ["flat", "cylindrical"])
@pytest.mark.parametrize("surfaces", [s for s in itertools.product([0, 1], repeat=4) if (s[0] or s[1]) and (s[2] or s[3])])
def test_corners(sfx, orc, sides, geometry, surfaces):
    bound = ["surface" if s else "mirror1" for s in surfaces]
    lat = LatticeSpec(2, sides, geometry=geometry, lowerbound=(bound[0], bound[2]), upperbound=(bound[1], bound[3]),
                      lambda_=0.2, offset_first_layer=1.5)
    wall = np.zeros(lat.dims[:2])
    for axis in (0, 1):
        for end in (0, 1):
            if surfaces[2 * axis + end]:
                wall[(slice(None),) * axis + (-end,)] = 1.0
    chi = np.array([[0, 0.5, 0.4, -0.6], [0.5, 0, 0.3, 0.2], [0.4, 0.3, 0, 0.1], [-0.6, 0.2, 0.1, 0]])
    sysd = SystemSpec(("A", "B", "S", "W"), chi, [MoleculeSpec("p", "(A)3(B)4", "free", phibulk=0.05),
                                                  MoleculeSpec("s", "(S)1", "solvent")], frozen={"W": wall.reshape(-1)})
    G, O = sfx.System(lat, sysd), orc.System(lat, sysd)
    x = np.random.default_rng(6).normal(0, 0.2, G.nvar)
    f, fo = G.residual(x), O.residual(x)
    assert np.abs(f - fo).max() <= 1e-11 * np.abs(fo).max()
    assert np.isfinite(O.free_energy())
    for a, b in ((G.free_energy(), O.free_energy()), (G.grand_potential(), O.grand_potential())):
        assert abs(a - b) <= 1e-11 * max(1.0, abs(b))
