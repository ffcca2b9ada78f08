"""Batched problems give the same bits at every number of threads per problem:
DIIS turns a last bit into another path, so a batch whose results followed the
tuner's choice could differ from the next one of the same problems. Lattices of
2 to 1024 layers, whose kernels hold one to seventeen layers per lane, problems
that converge and problems whose bulk is unstable."""
import numpy as np
import pytest

from field_amd import configs

pytestmark = pytest.mark.gpu

SMALL = [{"n_layers": n, "N": N, "chi_as": 0.3, "chi_s": -0.8, "phibulk": 0.02}
         for n in (2, 3, 9, 48, 49) for N in (2, 3, 18)]
LARGE = [{"n_layers": n, "N": 40, "chi_as": 0.9, "chi_s": -1.1, "phibulk": 0.01} for n in (97, 449, 897, 1024)]


@pytest.mark.parametrize("problems", [SMALL, SMALL + LARGE, configs.batch_1d(48)], ids=["small", "large", "uneven"])
def test_results_do_not_depend_on_the_threads(sfx, problems):
    B = sfx.Batch(problems)
    x = np.random.default_rng(3).normal(0, 0.1, B.nvar)
    ref = None
    for threads in (64, 128, 256, 512):
        B.set_threads(threads)
        assert B.tuning()[0] == threads
        f = B.residual(x)
        out = [f, B.lngn()] + [B.phi(i, s) for i in range(0, len(problems), 5) for s in (0, 1)]
        xs, its, norms, _ = B.solve(tolerance=1e-7, max_iter=400, diis_backtrack=1, diis_eta=1.0)
        out += [xs, its, norms]
        ref = ref or out
        for a, b in zip(out, ref):
            assert np.array_equal(a, b, equal_nan=True), threads


def test_other_numbers_of_threads_are_refused(sfx):
    B = sfx.Batch(SMALL[:2])
    for threads in (0, 32, 96, 1024):
        with pytest.raises(sfx.SFError):
            B.set_threads(threads)


def test_first_residual_of_a_batch_in_used_memory(sfx):
    """The store's surface entries are cleared before any launch reads them, also
    in memory that held something else: the first residual is the second's bits."""
    import torch

    x = None
    for _ in range(3):
        junk = torch.full((1 << 25,), float("nan"), dtype=torch.float64, device="cuda")
        del junk
        torch.cuda.empty_cache()
        B = sfx.Batch(configs.batch_1d(256))
        if x is None:
            x = np.random.default_rng(3).normal(0, 0.1, B.nvar)
            ref = B.residual(x)
        assert np.isfinite(ref).all() and np.array_equal(B.residual(x), ref)
        B.close()
