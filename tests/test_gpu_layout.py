"""The entry points' vectors are read and written by the kernels in their own
layout. Host and device vectors give the same bits, an output that overwrites an
input too, and a call leaves its x for those that need it later (the free energy
of the melt form), on every system of the parity set (1-D in one launch, 2-D,
3-D, second order, solids, melts).
"""
import numpy as np
import pytest
import torch

import cases
from field_amd import sfx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", cases.NAMES)
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_host_device_and_in_place(name, precision):
    lat, sysd = cases.case(name)
    x = cases.start(lat, sysd)
    v = np.random.default_rng(3).normal(0, 1, x.size)
    S = sfx.System(lat, sysd)
    f, jv = S.residual(x, precision=precision), S.jvp(x, v, precision=precision)
    F = S.free_energy()
    xd, vd = torch.from_numpy(x).cuda(), torch.from_numpy(v).cuda()
    S.residual(torch.zeros_like(xd), precision=precision)  # another x in between
    assert np.array_equal(S.residual(xd, precision=precision).cpu().numpy(), f)
    assert np.array_equal(S.jvp(xd, vd, precision=precision).cpu().numpy(), jv)
    assert S.free_energy() == F
    same = xd.clone()
    S.residual(same, precision=precision, out=same)
    assert np.array_equal(same.cpu().numpy(), f)
