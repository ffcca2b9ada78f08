"""Curved lattices with every pair of radial bounds, also those whose sweep is not
its own adjoint (mirror2, periodic): residuals against the oracle (sums of at
most 17 ranks' terms of one sign: 1e-12 of the largest entry), products against
its central difference (step 1e-5: 1e-10 of third derivatives of order 10 and
1e-16 / 1e-5 of rounding, 1e-7). Transposed products are refused where the sweep
is not its own adjoint, elsewhere w J v = v J^T w to the rounding of some 1400
terms, 1e-12 of the vectors' norms."""
import numpy as np
import pytest

from field_amd import _abi
from field_amd.spec import LatticeSpec, MoleculeSpec, SystemSpec

pytestmark = pytest.mark.gpu

RADIAL = [("mirror1", "mirror1"), ("mirror1", "surface"), ("surface", "mirror2"), ("mirror2", "mirror1"),
          ("mirror1", "mirror2"), ("mirror2", "mirror2"), ("periodic", "periodic")]


def lattice(name, radial):
    if name == "2d_cylinder":
        return LatticeSpec(2, (9, 51), geometry="cylindrical", lowerbound=(radial[0], "mirror1"),
                           upperbound=(radial[1], "mirror1"), lambda_=0.2, offset_first_layer=1.0)
    return LatticeSpec(1, (19,), geometry=name, lowerbound=radial[:1], upperbound=radial[1:], lambda_=0.2,
                       offset_first_layer=1.0)


@pytest.mark.parametrize("name", ["cylindrical", "spherical", "2d_cylinder"])
@pytest.mark.parametrize("radial", RADIAL)
@pytest.mark.parametrize("chain", ["(A)7(B)9", "(A)17"])
def test_bounds(sfx, orc, name, radial, chain):
    lat = lattice(name, radial)
    chi = np.array([[0, 0.5, 0.4], [0.5, 0, 0.3], [0.4, 0.3, 0]])
    sysd = SystemSpec(("A", "B", "S"), chi, [MoleculeSpec("p", chain, "restricted", theta=30.0), MoleculeSpec("s", "(S)1", "solvent")])
    G, O = sfx.System(lat, sysd), orc.System(lat, sysd)
    rng = np.random.default_rng(6)
    x, v = rng.normal(0, 0.2, G.nvar), rng.normal(0, 1, G.nvar)
    f, fo = G.residual(x), O.residual(x)
    assert np.abs(f - fo).max() <= 1e-12 * np.abs(fo).max()
    assert abs(G.lngn(0) - O.lngn(0)) <= 1e-12 * abs(O.lngn(0))
    jv = G.jvp(x, v)
    d = (O.residual(x + 1e-5 * v) - O.residual(x - 1e-5 * v)) / 2e-5
    assert np.abs(jv - d).max() <= 1e-7 * np.abs(d).max()
    w = rng.normal(0, 1, G.nvar)
    if "periodic" in radial or "mirror2" in radial:
        with pytest.raises(sfx.SFError) as e:
            G.vjp(x, w)
        assert e.value.code == _abi.SFX_E_UNSUPPORTED
    else:
        jtw = G.vjp(x, w)
        assert abs(w @ jv - jtw @ v) <= 1e-12 * np.linalg.norm(w) * np.linalg.norm(jv)
