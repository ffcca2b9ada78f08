"""Timed cases: the work that programs built on this library have it do.

Every case is one call (or, for the whole solves, one calculation) through the
public Python interface, `field_amd.sfx.System` / `Batch` and
`field_amd.torch_ops`, on device tensors, over the lattices, chain lengths,
boundary conditions and precisions of the repository's own workloads
(`field_amd.configs`) and tests:

  wall      homopolymer adsorption on a 1-D lattice (tens to a thousand layers)
  pore      diblock in a cylindrical pore, 2-D (r, z)
  melt      periodic simple-cubic diblock melt, 3-D
  mixture   3-D simple cubic with mirror bounds: triblock, homopolymer, solvent
  dense     3-D FCC / HEX, palindromic triblock in solvent
  semiflex  second-order (direction-resolved) homopolymer, 3-D
  batch     many uneven 1-D adsorption problems at once

`op` is what is asked of the system: `residual` f(u), `jvp` J v, `vjp`
(forward and backward of the torch function) or `solve`. Calls with FP32
sweeps hand their product on in FP32, the precision it has; FP64 sweeps give
FP64.
"""
import math

import numpy as np
import torch

from field_amd import configs, sfx, torch_ops
from field_amd.spec import LatticeSpec, MoleculeSpec, SystemSpec


# ---------------------------------------------------------------------------
# cases
def listed():
    return [
        # the smallest problem: one residual of 100 layers, as a caller with its own solver asks for it
        dict(name="wall_residual", family="wall", op="residual", precision="fp64", n=100, N=100),
        # Jacobian products of the same kind of problem (Newton-Krylov, gradients through a profile); odd sizes
        dict(name="wall_jvp", family="wall", op="jvp", precision="fp64", n=237, N=151),
        # a whole calculation with the default iteration from u = 0, parameters from a sweep
        dict(name="wall_newton", family="wall", op="solve", precision="fp64", n=100, N=100),
        # a parameter sweep: the residuals of uneven adsorption problems, evaluated together (an iteration of
        # the batched solve; the solve's own iterates depend on the last bit of every residual)
        dict(name="batch_residual", family="batch", op="residual", precision="fp64", count=512, n_max=400,
             N_max=1000),
        # 2-D: the residual of DIIS and the FP32 product of Newton-Krylov
        dict(name="pore_residual", family="pore", op="residual", precision="fp64", n=64, m=128, N=40),
        dict(name="pore_jvp", family="pore", op="jvp", precision="fp32", n=64, m=128, N=40),
        # the 64^3 melt: a whole chi sweep by Newton-Krylov
        dict(name="melt64_sweep", family="melt", op="solve", precision="fp32", n=64, m=64, k=64, N=40),
        # its FP32 product, the inner loop of that sweep
        dict(name="melt64_jvp", family="melt", op="jvp", precision="fp32", n=64, m=64, k=64, N=40),
        # the FP64 residual on a large box
        dict(name="melt128_residual", family="melt", op="residual", precision="fp64", n=128, m=128, k=128, N=40),
        # several molecules, mirror bounds and ragged sides; forward and backward of the torch function
        dict(name="mixture_vjp", family="mixture", op="vjp", precision="fp32", n=75, m=61, k=90, N=44),
        # twelve neighbours per site
        dict(name="fcc_residual", family="dense", op="residual", precision="fp64", n=50, m=41, k=63, N=40,
             lattice="fcc"),
        # the largest: direction-resolved chains with a quarter of the store's memory
        dict(name="semiflex_jvp", family="semiflex", op="jvp", precision="fp32", n=128, m=128, k=128, N=200,
             checkpointed=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["wall", "wall", "batch", "pore", "pore", "melt", "melt", "mixture", "dense", "semiflex"])
    op = rng.choice(["residual", "jvp", "vjp"])
    precision = rng.choice(["fp64", "fp32"])
    if family == "wall":
        op = rng.choice(["residual", "jvp", "solve"])
        n = _log_int(rng, 20, 1000 if op != "solve" else 150)
        return dict(family=family, op=op, precision=precision if op == "jvp" else "fp64", n=n,
                    N=_log_int(rng, 10, 500 if op != "solve" else 150))
    if family == "batch":
        return dict(family=family, op="residual", precision="fp64",
                    count=_log_int(rng, 32, 512), n_max=_log_int(rng, 60, 400), N_max=_log_int(rng, 40, 1000))
    if family == "pore":
        return dict(family=family, op=op, precision=precision, n=_log_int(rng, 8, 96), m=_log_int(rng, 8, 200),
                    N=2 * rng.randint(5, 40))
    if family == "melt":
        side = _log_int(rng, 12, 110)
        return dict(family=family, op=op, precision=precision, n=side, m=max(6, side + rng.randint(-5, 5)),
                    k=max(6, side + rng.randint(-5, 17)), N=rng.randint(12, 60))
    if family == "mixture":
        side = _log_int(rng, 10, 80)
        return dict(family=family, op=op, precision=precision, n=side, m=max(6, side + rng.randint(-5, 5)),
                    k=max(6, side + rng.randint(-5, 17)), N=rng.randint(16, 60))
    if family == "dense":
        side = _log_int(rng, 8, 64)
        return dict(family=family, op=rng.choice(["residual", "jvp"]), precision=precision, n=side,
                    m=max(5, side + rng.randint(-3, 5)), k=max(5, side + rng.randint(-3, 9)),
                    N=2 * rng.randint(6, 25), lattice=rng.choice(["fcc", "hex"]))
    side = _log_int(rng, 10, 80)
    return dict(family=family, op=op, precision=precision, n=side, m=max(6, side + rng.randint(-3, 3)),
                k=max(6, side + rng.randint(-3, 9)), N=rng.randint(12, 100), checkpointed=rng.random() < 0.5)


# ---------------------------------------------------------------------------
# the systems
def _chi(states, pairs):
    c = np.zeros((len(states), len(states)))
    for a, b, v in pairs:
        i, j = states.index(a), states.index(b)
        c[i, j] = c[j, i] = v
    return c


def _uniform(seed, n):
    return configs.uniform(1000 + seed, n)


def _system(case, seed):
    """(lattice, system) of a single-system case."""
    f, N = case["family"], case["N"]
    if f == "wall":
        par = dict(phibulk=0.01, chi_as=0.5, chi_s=-1.0)
        if case["op"] == "solve":  # a step of a parameter sweep
            u = _uniform(seed, 3)
            par = dict(phibulk=0.005 + 0.01 * u[0], chi_as=0.4 + 0.1 * u[1], chi_s=-1.1 + 0.2 * u[2])
        return configs.adsorption_1d(case["n"], N, **par)[:2]
    if f == "pore":
        lat, sysd, _ = configs.cylinder_2d(case["n"], case["m"])
        sysd.molecules[0] = MoleculeSpec("AB", f"(A){N // 2}(B){N - N // 2}", "free", phibulk=0.05)
        return lat, sysd
    sides = (case["n"], case["m"], case["k"])
    if f == "melt":
        a = max(1, round(0.3 * N))
        lat = LatticeSpec(3, sides, lowerbound=("periodic",) * 3, upperbound=("periodic",) * 3)
        sysd = SystemSpec(("A", "B"), np.array([[0.0, 0.4], [0.4, 0.0]]),
                          [MoleculeSpec("AB", f"(A){a}(B){N - a}", "restricted", theta=float(np.prod(sides)))],
                          form="melt", melt_phibulk=(0.0, 0.0))
        return lat, sysd
    if f == "mixture":
        lat = LatticeSpec(3, sides, lowerbound=("mirror1", "mirror2", "periodic"),
                          upperbound=("mirror2", "mirror1", "periodic"))
        st = ("A", "B", "S")
        a, c = N // 4, N // 5
        sysd = SystemSpec(st, _chi(st, [("A", "B", 0.8), ("A", "S", 0.4), ("B", "S", 0.6)]),
                          [MoleculeSpec("p", f"(A){a}(B){N - a - c}(A){c}", "restricted",
                                        theta=0.25 * float(np.prod(sides))),
                           MoleculeSpec("h", f"(B){N // 2 | 1}", "free", phibulk=0.1),
                           MoleculeSpec("s", "(S)1", "solvent")])
        return lat, sysd
    if f == "dense":
        lat = LatticeSpec(3, sides, lattice_type=case["lattice"], lowerbound=("periodic", "mirror1", "mirror2"),
                          upperbound=("periodic", "mirror1", "mirror1"))
        st = ("A", "B", "S")
        a = N // 4
        sysd = SystemSpec(st, _chi(st, [("A", "B", 0.7), ("A", "S", 0.2), ("B", "S", 0.9)]),
                          [MoleculeSpec("p", f"(A){a}(B){N - 2 * a}(A){a}", "restricted",
                                        theta=0.2 * float(np.prod(sides))),
                           MoleculeSpec("s", "(S)1", "solvent")])
        return lat, sysd
    lat = LatticeSpec(3, sides, order=2, lowerbound=("periodic",) * 3, upperbound=("periodic",) * 3)
    sysd = SystemSpec(("A", "S"), np.array([[0.0, 0.6], [0.6, 0.0]]),
                      [MoleculeSpec("pol", f"(A){N}", "restricted", theta=0.3 * float(np.prod(sides))),
                       MoleculeSpec("sol", "(S)1", "solvent")],
                      stiffness=1.0 / (1.0 + 4.0 * math.exp(-1.0)))
    return lat, sysd


def _problems(case, seed):
    """Uneven adsorption problems whose bulk is stable at any concentration (chi_as at most 1/2): the lattices and
    chains of a case are fixed, its chi parameters and bulk fractions come from the seed."""
    u = _uniform(seed, 5 * case["count"]).reshape(-1, 5)
    u[:, :2] = _uniform(0, 2 * case["count"]).reshape(-1, 2)
    lo, No = min(50, case["n_max"] // 2), min(20, case["N_max"] // 2)
    return [{"n_layers": lo + int(r[0] * (case["n_max"] - lo + 1)), "N": No + int(r[1] * (case["N_max"] - No + 1)),
             "chi_as": float(0.05 + 0.45 * r[2]), "chi_s": float(-1.2 * r[3]),
             "phibulk": float(10 ** (-4 + 3 * r[4]))} for r in u]


def _interior(lat):
    return tuple(lat.n_layers[: lat.gradients])


def _fields(case, seed):
    """(u, direction) of a system case: N(0, 0.1) fields around the bulk value 0 and an N(0, 1) direction, in
    the layout of the iteration vector."""
    lat, sysd = _system(case, seed)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    nv = sysd.n_itvar()
    out = []
    for sigma in (0.1, 1.0):
        if sysd.form == "melt":  # [state][padded lattice], halos 0
            v = torch.zeros((nv,) + lat.dims, dtype=torch.float64, device="cuda")
            inner = tuple(slice(1, n + 1) for n in _interior(lat))
            v[(slice(None),) + inner] = sigma * torch.randn((nv,) + _interior(lat), generator=gen, device="cuda",
                                                            dtype=torch.float64)
            out.append(v.reshape(-1))
        else:
            out.append(sigma * torch.randn(sysd.nvar(lat), generator=gen, device="cuda", dtype=torch.float64))
    return out


def prepare(case, seed):
    if case["family"] == "batch":
        batch = sfx.Batch(_problems(case, seed))
        gen = torch.Generator(device="cuda")
        gen.manual_seed(seed)
        x = 0.1 * torch.randn(batch.nvar, generator=gen, device="cuda", dtype=torch.float64)
        return dict(case=case, batch=batch, x=x)
    lat, sysd = _system(case, seed)
    budget = 0
    if case.get("checkpointed"):  # a quarter of the full store, but never below what checkpoints need
        ranks = max(case["N"] // 4, 3 * math.isqrt(case["N"]) + 3)
        budget = ranks * 6 * lat.M * 8
    system = sfx.System(lat, sysd, precision=case["precision"], memory_budget=budget)
    if case["family"] == "wall" and case["op"] == "solve":
        return dict(case=case, system=system, x=torch.zeros(system.nvar, dtype=torch.float64, device="cuda"))
    x, v = _fields(case, seed)
    return dict(case=case, system=system, x=x, v=v)


def run(state):
    case, x = state["case"], state["x"]
    op, precision = case["op"], case["precision"]
    if case["family"] == "batch":
        return state["batch"].residual(x)
    system = state["system"]
    if op == "solve":
        if case["family"] == "wall":
            xs, _ = system.solve(x, method="newton", tolerance=1e-7, max_iter=1000)
            return dict(x=xs, phi=[system.phi(0), system.phi(1)])
        # two steps of a chi sweep, the second from the first one's solution; the melt's fields are free up to
        # one constant, its volume fractions and its free energy are not
        system.solve_chi_sweep(x, 0, 1, [0.38, 0.4], method="nk", continuation=dict(ptc_dt0=0.0), tolerance=1e-9,
                               max_iter=60, gmres_rtol=0.3, jvp_precision=precision, ptc_dt0=3.0)
        return dict(phi=[system.phi(0), system.phi(1)], F=system.free_energy())
    if op == "residual":
        out = system.residual(x, precision=precision)
    elif op == "jvp":
        out = system.jvp(x, state["v"], precision=precision)
    else:
        u = x.detach().requires_grad_()
        f = torch_ops.residual(u, system, precision)
        (grad,) = torch.autograd.grad(f, u, state["v"])
        out = dict(f=f.detach(), grad=grad)
    if precision == "fp32":
        return {k: v.float() for k, v in out.items()} if isinstance(out, dict) else out.float()
    return out


# ---------------------------------------------------------------------------
# the work of a pass
def work(case):
    """The vectors in and out once, and the operations of the recursions: per site and rank a stencil and the
    segment weight for each of the two chains, and their composition; a tangent doubles both."""
    if case["family"] == "batch":
        n, N = (min(50, case["n_max"] // 2) + case["n_max"]) / 2, (min(20, case["N_max"] // 2) + case["N_max"]) / 2
        return {"bytes": 32.0 * n * case["count"], "flops": 8.0 * n * N * case["count"]}
    sites = case["n"] * case.get("m", 1) * case.get("k", 1)
    stencil = {"wall": 5, "pore": 8, "melt": 7, "mixture": 7, "dense": 13, "semiflex": 36}[case["family"]]
    ranks = case["N"] * (1.5 if case["family"] == "mixture" else 1.0)
    sweep = sites * ranks * (2 * stencil + (2 if case["family"] != "semiflex" else 12))
    half = 0.5 if case["family"] in ("wall", "dense") else 1.0  # a palindrome's backward chain is its forward chain
    base = sweep * half
    factor, vectors = {"residual": (1, 2), "jvp": (4, 3), "vjp": (5, 4),
                       "solve": (20 if case["family"] == "wall" else 40, 2)}[case["op"]]
    nv = 3 if case["family"] in ("pore", "mixture", "dense") else 2
    return {"bytes": 8.0 * vectors * nv * sites, "flops": base * factor}


# ---------------------------------------------------------------------------
# the same results in 64 bits with plain torch
def _shift(p, axis, d, lo, hi, edge):
    """Values at r + d (d = +-1) along an axis; beyond the ends the boundary's source layer, or `edge` (a number)
    behind a surface."""
    n = p.shape[axis]
    if d < 0:
        src = {"mirror1": 0, "mirror2": 1, "periodic": n - 1}.get(lo)
        end = p.narrow(axis, src, 1) if src is not None else torch.full_like(p.narrow(axis, 0, 1), edge)
        return torch.cat([end, p.narrow(axis, 0, n - 1)], axis)
    src = {"mirror1": n - 1, "mirror2": n - 2, "periodic": 0}.get(hi)
    end = p.narrow(axis, src, 1) if src is not None else torch.full_like(p.narrow(axis, 0, 1), edge)
    return torch.cat([p.narrow(axis, 1, n - 1), end], axis)


_HEX = [(-1, 0, 0), (1, 0, 0), (-1, 1, 0), (0, 1, 0), (0, -1, 0), (1, -1, 0), (0, 1, -1), (0, 0, -1), (1, 0, -1),
        (-1, 0, 1), (0, 0, 1), (0, -1, 1)]
_FCC = [(-1, -1, 0), (1, 1, 0), (-1, 1, 0), (1, -1, 0), (0, -1, -1), (0, 1, 1), (0, -1, 1), (0, 1, -1), (-1, 0, -1),
        (1, 0, 1), (-1, 0, 1), (1, 0, -1)]


def _average(lat, p, edge_x=(0.0, 0.0), contact=False):
    """The lattice average of a profile: of a propagator, or (contact) of a volume fraction; `edge_x`: its value
    in a surface layer below and above the first axis."""
    lo, hi, g = lat.lowerbound, lat.upperbound, lat.gradients

    def at(*ds):
        q = p
        for axis, d in enumerate(ds):
            if d:
                q = _shift(q, axis, d, lo[axis], hi[axis], edge_x[0 if d < 0 else 1] if axis == 0 else 0.0)
        return q

    if g == 1:
        return p + lat.lambda_ * (at(-1) - 2 * p + at(1))
    if g == 2:
        i = torch.arange(1, p.shape[0] + 1, dtype=p.dtype, device=p.device).reshape(-1, 1)
        lm, lp = lat.lambda_ * 2 * (i - 1) / (2 * i - 1), lat.lambda_ * 2 * i / (2 * i - 1)
        return (p + lm * (at(-1, 0) - p) + lp * (at(1, 0) - p) + lat.lambda_ * (at(0, -1) + at(0, 1) - 2 * p))
    if lat.lattice_type == "fcc" and contact:
        rows = at(-1, 0, 0) + p + at(1, 0, 0)
        p = rows
        rows = at(0, -1, 0) + p + at(0, 1, 0)
        p = rows
        return (at(0, 0, -1) + p + at(0, 0, 1)) / 27.0
    steps = {"fcc": _FCC, "hex": _HEX, "standard": [(-1, 0, 0), (1, 0, 0), (0, -1, 0), (0, 1, 0), (0, 0, -1),
                                                    (0, 0, 1)]}[lat.lattice_type]
    s = 0
    for d in steps:
        s = s + at(*d)
    return s / len(steps)


def _weights(lat, like):
    """Weight of a site in the partition function: 1, 1/2 in a mirror2 layer, the ring's area in a cylinder."""
    w = torch.ones_like(like)
    for k in range(lat.gradients):
        if lat.lowerbound[k] == "mirror2":
            w.narrow(k, 0, 1).mul_(0.5)
        if lat.upperbound[k] == "mirror2":
            w.narrow(k, w.shape[k] - 1, 1).mul_(0.5)
    if lat.gradients == 2:
        i = torch.arange(1, like.shape[0] + 1, dtype=like.dtype, device=like.device).reshape(-1, 1)
        w = w * math.pi * (2 * i - 1)
    return w


_E = [(0, 1), (1, 1), (2, 1), (2, -1), (1, -1), (0, -1)]  # bond directions +x, +y, +z, -z, -y, -x


def _chain(lat, sysd, g, seq):
    """(unnormalised composition per state, sum of the end ranks) of one chain."""
    N, acc = len(seq), {}
    if lat.order == 1:
        fwd = [g[seq[0]]]
        for s in range(1, N):
            fwd.append(g[seq[s]] * _average(lat, fwd[-1]))
        end = (_weights(lat, g[0]) * fwd[-1]).sum()
        b = g[seq[-1]]
        for s in range(N - 1, -1, -1):
            if s < N - 1:
                b = g[seq[s]] * _average(lat, b)
            acc[seq[s]] = acc.get(seq[s], 0) + fwd.pop() * b
        return {t: a / g[t] for t, a in acc.items()}, end
    S = sysd.stiffness
    L = (1 - S) / 4

    def transfer(G):
        return S * G + L * (G.sum(0, keepdim=True) - G - G.flip(0))

    def step_f(G, gt):
        W = transfer(G)
        return torch.stack([gt * torch.roll(W[k], d, a) for k, (a, d) in enumerate(_E)])

    def step_b(G, gt):
        return gt * transfer(torch.stack([torch.roll(G[k], -d, a) for k, (a, d) in enumerate(_E)]))

    fwd = [g[seq[0]].expand(6, *g[0].shape)]
    for s in range(1, N):
        fwd.append(step_f(fwd[-1], g[seq[s]]))
    end = fwd[-1].sum() / 6
    b = g[seq[-1]].expand(6, *g[0].shape)
    for s in range(N - 1, -1, -1):
        if s < N - 1:
            b = step_b(b, g[seq[s]])
        acc[seq[s]] = acc.get(seq[s], 0) + (fwd.pop() * b).sum(0) / 6
    return {t: a / g[t] for t, a in acc.items()}, end


def _residual64(lat, sysd, u):
    """f(u) on interior arrays: u and f are (variables, *sides); every liquid state has its own variable here."""
    states, chi = list(sysd.states), np.asarray(sysd.chi)
    liquid = [i for i, s in enumerate(states) if s not in sysd.frozen]
    var = {t: k for k, t in enumerate(liquid)}
    g = {t: torch.exp(-u[var[t]]) for t in liquid}
    phi = {t: 0 for t in liquid}
    bulk = {t: 0.0 for t in range(len(states))}
    left = 1.0
    for m, seq in sorted(zip(sysd.molecules, sysd.sequences()), key=lambda z: z[0].freedom == "solvent"):
        N = len(seq)
        if N == 1:
            comp, end = {seq[0]: g[seq[0]]}, (_weights(lat, g[seq[0]]) * g[seq[0]]).sum()
        else:
            comp, end = _chain(lat, sysd, g, seq)
        if m.freedom == "restricted":
            phib, c = m.theta / end, m.theta / (N * end)
        else:
            phib = m.phibulk if m.freedom == "free" else left
            c = phib / N
        left = left - phib
        for t, p in comp.items():
            phi[t] = phi[t] + c * p
            bulk[t] = bulk[t] + phib * (seq.count(t) / N)
    if sysd.form == "melt":
        bulk = dict(enumerate(sysd.melt_phibulk))
    total = sum(phi.values())
    rho = {t: _average(lat, phi[t], contact=True) for t in liquid}
    for t, s in enumerate(states):
        if s in sysd.frozen:  # a wall in a surface layer of the first axis, seen from the layer next to it
            prof = np.asarray(sysd.frozen[s]).reshape(lat.dims)
            edge = (float(prof[0].reshape(-1)[1 if prof[0].size > 1 else 0]),
                    float(prof[-1].reshape(-1)[1 if prof[-1].size > 1 else 0]))
            rho[t] = _average(lat, torch.zeros_like(u[0]), edge, contact=True)
    up = []
    for t in liquid:
        v = u[var[t]]
        for j in range(len(states)):
            if chi[t, j]:
                v = v - chi[t, j] * rho[j] / total
                if states[j] not in sysd.frozen:
                    v = v + chi[t, j] * bulk[j]
        up.append(v)
    mean = sum(up) / len(up)
    return torch.stack([-1.0 + 1.0 / total + v - mean for v in up])


def _batch64(problems, x):
    """The residuals of all problems side by side, each row padded to the longest lattice and chain."""
    n = torch.tensor([p["n_layers"] for p in problems], device=x.device)
    N = torch.tensor([p["N"] for p in problems], device=x.device)
    B, width, ranks = len(problems), int(n.max()), int(N.max())
    layer = torch.arange(width, device=x.device)
    inside = layer[None, :] < n[:, None]
    last = layer[None, :] == n[:, None] - 1
    u = torch.zeros(B, width, 2, dtype=x.dtype, device=x.device)
    u[inside] = x.reshape(-1, 2)
    col = {k: torch.tensor([p[k] for p in problems], dtype=x.dtype, device=x.device)[:, None]
           for k in ("chi_as", "chi_s", "phibulk")}
    g = torch.exp(-u) * inside[..., None]

    def average(p):  # 0 in the surface layer below, mirrored above
        down = torch.cat([torch.zeros_like(p[:, :1]), p[:, :-1]], 1)
        up = torch.where(last, p, torch.cat([p[:, 1:], torch.zeros_like(p[:, :1])], 1))
        return (p + (down - 2 * p + up) / 6.0) * inside

    G = torch.empty(ranks, B, width, dtype=x.dtype, device=x.device)
    G[0] = g[..., 0]
    for s in range(1, ranks):
        G[s] = g[..., 0] * average(G[s - 1])
    phi = torch.zeros_like(g)
    row = torch.arange(B, device=x.device)
    for s in range(ranks):  # the homopolymer's backward chain is its forward chain
        partner = G[(N - 1 - s).clamp(min=0), row]
        phi[..., 0] += torch.where((s < N)[:, None], G[s] * partner, torch.zeros_like(partner))
    g_in = torch.where(inside[..., None], g, torch.ones_like(g))
    phi[..., 0] *= col["phibulk"] / N[:, None] / g_in[..., 0]
    phi[..., 1] = (1 - col["phibulk"]) * g[..., 1]
    total = torch.where(inside, phi.sum(-1), torch.ones_like(phi[..., 0]))
    wall = torch.zeros_like(total)
    wall[:, 0] = 1.0 / 6.0
    vA = u[..., 0] - (col["chi_as"] * average(phi[..., 1]) + col["chi_s"] * wall) / total + col["chi_as"] * (
        1 - col["phibulk"])
    vS = u[..., 1] - col["chi_as"] * average(phi[..., 0]) / total + col["chi_as"] * col["phibulk"]
    mean = 0.5 * (vA + vS)
    return torch.stack([-1 + 1 / total + vA - mean, -1 + 1 / total + vS - mean], -1)[inside].reshape(-1)


def exact(case, seed):
    if case["family"] == "batch":
        return _batch64(_problems(case, seed), prepare(case, seed)["x"])
    lat, sysd = _system(case, seed)
    if case["op"] == "solve":
        if case["family"] != "melt":
            return None
        # below the spinodal the melt's solution is homogeneous: phi_A = f_A everywhere (halo layers included)
        N, V, fa = case["N"], float(np.prod(_interior(lat))), round(0.3 * case["N"]) / case["N"]
        return dict(phi=[np.full(lat.M, fa), np.full(lat.M, 1 - fa)], F=0.4 * V * fa * (1 - fa))
    x, v = _fields(case, seed)
    sides, nv = _interior(lat), sysd.n_itvar()
    melt = sysd.form == "melt"
    inner = (slice(None),) + tuple(slice(1, n + 1) for n in sides)

    def split(q):
        return q.reshape((nv,) + lat.dims)[inner] if melt else torch.movedim(q.reshape(sides + (nv,)), -1, 0)

    def join(q):
        if not melt:
            return torch.movedim(q, 0, -1).reshape(-1)
        out = torch.zeros((nv,) + lat.dims, dtype=q.dtype, device=q.device)
        out[inner] = q
        return out.reshape(-1)

    def f(q):
        return _residual64(lat, sysd, q)

    if case["op"] == "residual":
        return join(f(split(x)))
    if case["op"] == "jvp":
        return join(torch.func.jvp(f, (split(x),), (split(v),))[1])
    u = split(x).clone().requires_grad_()
    val = f(u)
    (grad,) = torch.autograd.grad(val, u, split(v))
    return dict(f=join(val.detach()), grad=join(grad))
