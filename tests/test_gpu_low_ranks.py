"""FP32 sweeps of several ranks per launch where a chain's weight lies far from
the lattice maximum of g: a site of u = 0 in a lattice of u = depth, on lattices
whose step gives a site no weight of its own, so that two ranks lose the factor
exp(-depth). A launch renormalises only its input; from some 17 kT within one
launch on the evaluation is repeated rank by rank, so every depth has to give
the FP64 result: rounding of 1e-7 per rank over at most 41 ranks, 2e-5 of the
largest entry. Depths below and above that line, and ones at which the ranks of
a launch reach FP32's smallest numbers. A second polymer, without a field, fills
the lattice. Strong noise reaches FP32's range in every kernel: there the blocked
sweeps may be no further off than four times the per-rank ones, or 2e-5.
"""
import numpy as np
import pytest
import torch

from field_amd.spec import LatticeSpec, MoleculeSpec, SystemSpec

pytestmark = pytest.mark.gpu

LATTICES = {"2d": LatticeSpec(2, (24, 60), lowerbound=("periodic",) * 2, upperbound=("periodic",) * 2, lambda_=0.25),
            "sc": LatticeSpec(3, (12, 11, 18), lowerbound=("periodic",) * 3, upperbound=("periodic",) * 3),
            "fcc": LatticeSpec(3, (12, 11, 18), lattice_type="fcc", lowerbound=("periodic",) * 3,
                               upperbound=("periodic",) * 3)}
CHAINS = ["(A)20(B)21", "(A)40", "(A)41"]


def system(lattice, chain):
    lat = LATTICES[lattice]
    chi = np.array([[0.0, 0.8, 0.4], [0.8, 0.0, 0.6], [0.4, 0.6, 0.0]])
    return lat, SystemSpec(("A", "B", "C"), chi,
                           [MoleculeSpec("p", chain, "restricted", theta=2.0),
                            MoleculeSpec("c", "(C)7", "restricted", theta=float(np.prod(lat.n_layers)))],
                           form="melt", melt_phibulk=(0.0, 0.0, 0.0))


def fields(lat, sysd, depth):
    """A well for A and B, and a direction; the layout [state][padded lattice]."""
    interior = (slice(None),) + tuple(slice(1, n + 1) for n in lat.n_layers)
    dims = (3,) + tuple(n + 2 for n in lat.n_layers)
    u, w = np.zeros(dims), np.zeros(dims)
    u[interior][:2] = depth
    u[(slice(None),) + tuple(1 + n // 2 for n in lat.n_layers)] = 0.0
    w[interior] = np.random.default_rng(1).normal(0, 1, w[interior].shape)
    return u.reshape(-1), w.reshape(-1)


def close(a, b):
    return np.isfinite(b).all() and np.abs(a - b).max() <= 2e-5 * np.abs(b).max()


@pytest.mark.parametrize("lattice", LATTICES)
@pytest.mark.parametrize("chain", CHAINS)
@pytest.mark.parametrize("depth", [4, 8, 10, 13, 16, 20, 24, 28])
def test_deep_site(sfx, lattice, chain, depth):
    print(lattice, chain, depth, flush=True)
    lat, sysd = system(lattice, chain)
    G = sfx.System(lat, sysd)
    x, w = fields(lat, sysd, depth)
    for what in ("residual", "jvp", "vjp"):
        arg = (x,) if what == "residual" else (x, w)
        a = getattr(G, what)(*arg, precision="fp32")
        phi, lngn = G.phi(0), G.lngn(0)
        b = getattr(G, what)(*arg)
        assert close(a, b), what
        assert close(phi, G.phi(0)) and abs(lngn - G.lngn(0)) <= 1e-5, what


@pytest.mark.parametrize("chain", CHAINS)
@pytest.mark.parametrize("options", [dict(chain_schedule="sequential"), dict(memory_budget=20 * 8 * LATTICES["sc"].M)],
                         ids=["sequential", "checkpointed"])
def test_other_schedules(sfx, chain, options):
    lat, sysd = system("sc", chain)
    G, P = sfx.System(lat, sysd, **options), sfx.System(lat, sysd, sweep_kernel="per_rank")
    x, w = fields(lat, sysd, 24)
    assert np.array_equal(G.residual(x, precision="fp32"), P.residual(x, precision="fp32"))
    assert np.array_equal(G.jvp(x, w, precision="fp32"), P.jvp(x, w, precision="fp32"))
    assert np.array_equal(G.vjp(x, w, precision="fp32"), P.vjp(x, w, precision="fp32"))


@pytest.mark.parametrize("chain", CHAINS)
def test_results_over_the_inputs(sfx, chain):
    """A repeated evaluation takes its inputs from where the first pass has not written."""
    lat, sysd = system("2d", chain)
    G = sfx.System(lat, sysd)
    x, w = (torch.from_numpy(a).cuda() for a in fields(lat, sysd, 24))
    f, jv = G.residual(x, precision="fp32"), G.jvp(x, w, precision="fp32")
    ptr = lambda a: sfx._ptr(a)[0]
    a, b = x.clone(), w.clone()
    sfx.check(sfx.lib().sfx_jvp(G.h, ptr(a), ptr(b), ptr(b), 1, 1))
    assert torch.equal(b, jv)
    b = w.clone()
    sfx.check(sfx.lib().sfx_jvp(G.h, ptr(a), ptr(b), ptr(a), 1, 1))
    assert torch.equal(a, jv)
    a = x.clone()
    G.residual(a, precision="fp32", out=a)
    assert torch.equal(a, f)


@pytest.mark.parametrize("lattice", ["2d", "sc"])
@pytest.mark.parametrize("chain", CHAINS)
def test_newton_krylov_steps(sfx, lattice, chain):
    """Two steps of a solve whose first sweeps decay too far: the solve goes on
    rank by rank, as one that was rank by rank from its start."""
    lat, sysd = system(lattice, chain)
    x, _ = fields(lat, sysd, 24)
    opts = dict(method="nk", check_converged=False, max_iter=2, tolerance=1e-9, ptc_dt0=0.0, precondition=0)
    a, sa = sfx.System(lat, sysd).solve(x, **opts)
    b, sb = sfx.System(lat, sysd, sweep_kernel="per_rank").solve(x, **opts)
    assert sa["iterations"] == sb["iterations"] == 2 and sa["residual_evals_fp32"] > 0
    assert close(a, b)
    # and the next evaluation of an ordinary field is by blocked launches again
    G = sfx.System(lat, sysd)
    y = 0.01 * x
    f = G.residual(y, precision="fp32")
    G.solve(x, **opts)
    assert np.array_equal(G.residual(y, precision="fp32"), f)


@pytest.mark.parametrize("lattice", LATTICES)
@pytest.mark.parametrize("sigma", [0.5, 1.0, 1.5])
@pytest.mark.parametrize("seed", range(4))
def test_strong_noise(sfx, lattice, sigma, seed):
    """Also of a molecule whose amount is fixed in a box that its weight avoids."""
    lat = LATTICES[lattice]
    chi = np.array([[0.0, 0.8, 0.4], [0.8, 0.0, 0.6], [0.4, 0.6, 0.0]])
    far = tuple(max(1, n // 4) for n in lat.n_layers) + (1,) * (3 - len(lat.n_layers))
    box = MoleculeSpec("b", "(A)26", "range_restricted", range_lo=far, range_hi=far, phi_range=1.0)
    for molecules, products in (([MoleculeSpec("p", "(A)20(B)21", "restricted", theta=9.0)], True), ([box], False)):
        sysd = SystemSpec(("A", "B", "S"), chi, molecules + [MoleculeSpec("q", "(B)9", "free", phibulk=0.05),
                                                             MoleculeSpec("s", "(S)1", "solvent")])
        G, P = sfx.System(lat, sysd), sfx.System(lat, sysd, sweep_kernel="per_rank")
        rng = np.random.default_rng(seed)
        x, w = rng.normal(0, sigma, G.nvar), rng.normal(0, 1, G.nvar)
        for what in ("residual", "jvp", "vjp") if products else ("residual",):
            arg = (x,) if what == "residual" else (x, w)
            ref = getattr(G, what)(*arg)
            a, b = (np.abs(getattr(S, what)(*arg, precision="fp32") - ref).max() for S in (G, P))
            assert a <= max(4 * b, 2e-5 * np.abs(ref).max()) or not np.isfinite(b), (what, a, b)


def test_a_refused_call_leaves_nothing_behind(sfx):
    """A product that is refused after its sweep has found low ranks: the next
    evaluation, of an ordinary field, is by blocked launches, to the same bits."""
    lat = LATTICES["2d"]
    box = MoleculeSpec("b", "(A)26", "range_restricted", range_lo=(6, 15, 1), range_hi=(9, 20, 1), phi_range=1.0)
    sysd = SystemSpec(("A", "S"), np.array([[0.0, 0.4], [0.4, 0.0]]), [box, MoleculeSpec("s", "(S)1", "solvent")])
    G = sfx.System(lat, sysd)
    rng = np.random.default_rng(2)
    x, steep = rng.normal(0, 0.1, G.nvar), rng.normal(0, 3.0, G.nvar)
    f = G.residual(x, precision="fp32")
    with pytest.raises(sfx.SFError):
        G.jvp(steep, x, precision="fp32")
    assert np.array_equal(G.residual(x, precision="fp32"), f)
    P = sfx.System(lat, sysd, sweep_kernel="per_rank")  # the two paths can be told apart
    assert not np.array_equal(P.residual(x, precision="fp32"), f)
