"""The transposed product's sums and coefficients, made on the device, on
lattices of less than one wave to several hundred workgroups, with molecules of
every freedom (two restricted, one free, a solvent), monomers and chains: the
transposed product is the transpose, <w, J v> = <J^T w, v>. Both sides round at
1e-16 of their terms' norms, over a few ranks and sums of up to 3e5 terms: 1e-11
of |w| |J v|.
"""
import numpy as np
import pytest

from field_amd import sfx
from field_amd.spec import LatticeSpec, MoleculeSpec, SystemSpec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sides", [(5, 7), (16, 16), (23, 45), (300, 340)])
@pytest.mark.parametrize("solvent", ["(S)1", "(S)2"])
def test_transpose(sides, solvent):
    print(sides, solvent, flush=True)
    lat = LatticeSpec(2, sides, lowerbound=("mirror2", "periodic"), upperbound=("mirror1", "periodic"), lambda_=0.2)
    chi = np.array([[0.0, 0.8, 0.4], [0.8, 0.0, 0.6], [0.4, 0.6, 0.0]])
    n = float(np.prod(sides))
    sysd = SystemSpec(("A", "B", "S"), chi,
                      [MoleculeSpec("p", "(A)3(B)4", "restricted", theta=0.2 * n),
                       MoleculeSpec("q", "(B)1", "restricted", theta=0.1 * n),
                       MoleculeSpec("h", "(B)3(A)1", "free", phibulk=0.1), MoleculeSpec("s", solvent, "solvent")])
    rng = np.random.default_rng(5)
    nv = sysd.nvar(lat)
    x, v, w = rng.normal(0, 0.1, nv), rng.normal(0, 1, nv), rng.normal(0, 1, nv)
    S = sfx.System(lat, sysd)
    jv, jw = S.jvp(x, v, precision="fp64"), S.vjp(x, w, precision="fp64")
    assert abs(w @ jv - jw @ v) <= 1e-11 * np.linalg.norm(w) * np.linalg.norm(jv)
    assert np.array_equal(S.vjp(x, w, precision="fp64"), jw)
