"""Local energies of the transverse-field Ising model by small ResConvs (a candidate per
site, one wave each on one and two tiles) against the oracle.  Tolerances of the other
ResConv tests: 1e-5 (FP32), 1e-4 (split-bf16) relative with a floor of 1."""
import numpy as np
import pytest
import torch

from oracle import models as om
from oracle import operator as oop
from tests.helpers import max_rel, rand_spins

pytestmark = pytest.mark.gpu

import quantax_amd as qtx  # noqa: E402


@pytest.mark.parametrize("L0,L1", [(1, 2), (2, 2), (3, 5), (4, 4), (1, 17), (3, 9), (4, 8), (3, 11)])
@pytest.mark.parametrize("C,prec,tol", [(16, "fp32", 1e-5), (16, "bf16x3", 1e-4), (32, "fp32", 1e-5)])
def test_ising(L0, L1, C, prec, tol):
    rng = np.random.default_rng(L0 + 7 * L1)
    N = L0 * L1
    qtx.sites.Grid([L0, L1])
    model = qtx.model.ResConv(1, C, precision=prec, seed=8)
    H, Ho = qtx.operator.Ising(h=1.0), oop.ising([L0, L1], 1.0)
    s = rand_spins(rng, 70, N)
    sd = torch.from_numpy(s).cuda()
    la = model.logpsi(sd)
    e, nc = model.eloc(H, sd, la)
    theta, spec = model.theta.cpu().numpy().astype(np.float64), om.ResConvSpec(1, C, (L0, L1))
    ref = oop.oloc(s[:3], lambda x: om.resconv_forward(spec, theta, x), Ho)
    assert max_rel(e[:3].cpu().numpy(), ref) < tol
    assert bool((nc == N).all())
    for i in (0, 33, 69):
        e1, _ = model.eloc(H, sd[i: i + 1], la[i: i + 1])
        assert abs(float(e1[0] - e[i])) <= 1e-12 * max(1.0, abs(float(e[i]))) * 4
