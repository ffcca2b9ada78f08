"""Calls that find no memory for the buffers they keep: each is refused with
SFX_E_OOM, so is the next one, what needs no new memory still runs, and once
memory is there every call gives what a fresh system gives."""
import gc

import numpy as np
import pytest
import torch

from field_amd import _abi
from field_amd.spec import LatticeSpec, MoleculeSpec, SystemSpec

pytestmark = pytest.mark.gpu


def system(sides, lattice_type="standard"):
    lat = LatticeSpec(3, sides, lattice_type=lattice_type, lowerbound=("periodic",) * 3, upperbound=("periodic",) * 3)
    chi = np.array([[0.0, 0.5, 0.4], [0.5, 0.0, 0.3], [0.4, 0.3, 0.0]])
    return lat, SystemSpec(("A", "B", "S"), chi, [MoleculeSpec("p", "(A)9(B)8", "restricted", theta=0.2 * float(np.prod(sides))),
                                                  MoleculeSpec("s", "(S)1", "solvent")])


def calls(G, x, v):
    opts = dict(max_iter=2, check_converged=False)
    return {"jvp": lambda: G.jvp(x, v), "vjp": lambda: G.vjp(x, v),
            "diis": lambda: G.solve(x, diis_m=10, **opts)[0],
            "nk": lambda: G.solve(x, method="nk", gmres_restart=20, **opts)[0]}


def inputs(nvar):
    rng = np.random.default_rng(5)
    return rng.normal(0, 0.05, nvar), rng.normal(0, 1, nvar)


class Filled:
    """The device's memory taken but for `most` bytes; leave(n) takes all but n of
    what is free then."""

    def __init__(self, most):
        self.most, self.more = most, None

    def __enter__(self):
        gc.collect()
        torch.cuda.empty_cache()
        free, _ = torch.cuda.mem_get_info()
        self.hold = torch.empty(free - self.most, dtype=torch.uint8, device="cuda")
        return self

    def leave(self, n):
        self.more = []
        torch.cuda.empty_cache()
        for _ in range(8):  # what a large allocation really takes is known after it
            free, _ = torch.cuda.mem_get_info()
            if free - n < 4 << 20:
                return
            self.more.append(torch.empty(free - n, dtype=torch.uint8, device="cuda"))

    def __exit__(self, *_):
        self.hold = self.more = None
        torch.cuda.empty_cache()


def test_refused_twice_and_served_later(sfx):
    small = system((12, 12, 20))
    S = sfx.System(*small)
    for run in calls(S, *inputs(S.nvar)).values():  # what the runtime sets up once per kernel
        run()
    lat, sysd = system((110, 110, 110))  # 11 MiB an array, 31 MiB a vector
    x, v = inputs(sysd.nvar(lat))
    fresh = sfx.System(lat, sysd)
    ref = {name: run() for name, run in calls(fresh, x, v).items()}
    fresh.close()
    systems = {left: sfx.System(lat, sysd) for left in (320, 128, 64)}
    f = [G.residual(x) for G in systems.values()]
    with Filled(2 << 30) as memory:
        for left, G in systems.items():
            memory.leave(left << 20)
            refused = []
            for _ in range(2):
                for name, run in calls(G, x, v).items():
                    try:
                        run()
                    except sfx.SFError as e:
                        assert e.code == _abi.SFX_E_OOM, name
                        refused.append(name)
                    assert np.array_equal(G.residual(x), f[0]), name
            print(left, refused, flush=True)
            assert refused
    for G in systems.values():
        for name, run in calls(G, x, v).items():
            assert np.array_equal(run(), ref[name]), name


def used():
    free, total = torch.cuda.mem_get_info()
    return total - free


def test_fcc_fits_where_it_fitted_rank_by_rank(sfx):
    """The second accumulators of blocked FCC sweeps are left out, or given back,
    where they do not fit; the system is then swept rank by rank."""
    lat, sysd = system((120, 120, 120), "fcc")  # 14 MiB an array; second accumulators and ranks 111 MiB
    x, v = inputs(sysd.nvar(lat))
    for lattice in (lat, system((9, 9, 9), "fcc")[0]):  # the kernels of both paths have run once
        for kernel in ("auto", "per_rank"):
            S = sfx.System(lattice, sysd, sweep_kernel=kernel)
            xs, vs = inputs(S.nvar)
            S.jvp(xs, vs), S.vjp(xs, vs), S.residual(xs)
            S.close()
    gc.collect()
    torch.cuda.empty_cache()
    u0 = used()
    P = sfx.System(lat, sysd, sweep_kernel="per_rank")
    need = used() - u0
    f = P.residual(x)
    u1 = used()
    jv = P.jvp(x, v)
    tangents = used() - u1
    jtw = P.vjp(x, v)
    P.close()
    assert tangents > 200 << 20
    with Filled(2 << 30) as memory:
        memory.leave(need + (40 << 20))
        G = sfx.System(lat, sysd)
        assert np.array_equal(G.residual(x), f)
        G.close()
    G = sfx.System(lat, sysd)
    assert np.abs(G.residual(x) - f).max() <= 1e-12 * np.abs(f).max()
    with Filled(2 << 30) as memory:
        memory.leave(tangents - (50 << 20))
        assert np.array_equal(G.jvp(x, v), jv)
        assert np.array_equal(G.residual(x), f)
    assert np.array_equal(G.vjp(x, v), jtw)
