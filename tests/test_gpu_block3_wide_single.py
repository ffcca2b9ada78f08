"""FP32 base launches of one chain on the tile of 16 planes (from 896 workgroups
of the smaller tile on): palindromes, sequential schedules and checkpointed
stores against the one-launch-per-rank kernels, FP32 rounding of 1e-7 per rank
over 41 ranks in both, 2e-5 of the largest entry. A checkpointed store repeats
its stretches by the launches of the first pass, so it gives the bits of the
full one."""
import numpy as np
import pytest

from field_amd import sfx
from field_amd.spec import LatticeSpec, MoleculeSpec, SystemSpec

pytestmark = pytest.mark.gpu

SIDES = (113, 61, 130)


@pytest.mark.parametrize("chain,slots", [("(A)20(B)21", 20), ("(A)15(B)11(A)15", 18), ("(A)40", 18)])
def test_single_chains(chain, slots):
    assert -(-SIDES[0] // 8) * -(-SIDES[1] // 8) * -(-SIDES[2] // 16) >= 896
    lat = LatticeSpec(3, SIDES, lowerbound=("mirror1", "mirror2", "periodic"),
                      upperbound=("mirror2", "mirror1", "periodic"))
    chi = np.array([[0.0, 0.8, 0.4], [0.8, 0.0, 0.6], [0.4, 0.6, 0.0]])
    sysd = SystemSpec(("A", "B", "S") if "B" in chain else ("A", "S"), chi if "B" in chain else chi[::2, ::2],
                      [MoleculeSpec("p", chain, "restricted", theta=0.3 * float(np.prod(SIDES))),
                       MoleculeSpec("s", "(S)1", "solvent")])
    x = np.random.default_rng(4).normal(0, 0.2, sysd.nvar(lat))
    f = {}
    for name, opts in {"auto": {}, "sequential": dict(chain_schedule="sequential"),
                       "checkpointed": dict(memory_budget=slots * 8 * lat.M), "per_rank": dict(sweep_kernel="per_rank")}.items():
        G = sfx.System(lat, sysd, **opts)
        f[name] = G.residual(x, precision="fp32")
        G.close()
    for name in ("auto", "sequential", "checkpointed"):
        assert np.abs(f[name] - f["per_rank"]).max() <= 2e-5 * np.abs(f["per_rank"]).max(), name
    assert np.array_equal(f["checkpointed"], f["sequential"])
