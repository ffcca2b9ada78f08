"""The wider tile (16 x 8 x 16 sites) of FP32 base ranks on large simple cubic
lattices, at x sides around it, against the one-launch-per-rank kernels: FP32
rounding of 1e-7 per rank over at most 21 ranks in both, 2e-5 of the largest
entry."""
import numpy as np
import pytest

from field_amd import sfx
from field_amd.spec import LatticeSpec, MoleculeSpec, SystemSpec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx", [63, 64, 65, 73])
@pytest.mark.parametrize("n", [5, 10])
def test_wide_tile_matches_per_rank(nx, n):
    sides = (nx, 61, 130)  # 896 workgroups of the smaller tile, or more, for two chains
    assert 2 * -(-nx // 8) * 8 * 9 >= 896
    lat = LatticeSpec(3, sides, lowerbound=("mirror1", "mirror2", "periodic"),
                      upperbound=("mirror2", "mirror1", "periodic"))
    chi = np.array([[0.0, 0.8, 0.4], [0.8, 0.0, 0.6], [0.4, 0.6, 0.0]])
    sysd = SystemSpec(("A", "B", "S"), chi,
                      [MoleculeSpec("p", f"(A){n}(B){n + 1}", "restricted", theta=0.3 * float(np.prod(sides))),
                       MoleculeSpec("s", "(S)1", "solvent")])
    x = np.random.default_rng(4).normal(0, 0.2, sysd.nvar(lat))
    a = sfx.System(lat, sysd).residual(x, precision="fp32")
    b = sfx.System(lat, sysd, sweep_kernel="per_rank").residual(x, precision="fp32")
    assert np.abs(a - b).max() <= 2e-5 * np.abs(b).max()
