"""The any-lattice ResConv kernels at the edges of their classes (needs an
MI355X): lattices of 1 to 32 tiles with and without a ragged last one, few and
many configurations (four, two or one waves each), against the oracle, and the
amplitudes of one configuration the same bit for bit whichever class evaluates
it.  Tolerances of the other ResConv tests: 1e-5 (FP32), 1e-4 (split-bf16)
relative with a floor of 1."""
import numpy as np
import pytest
import torch

from oracle import models as om
from oracle import operator as oop
from tests.helpers import max_rel, rand_spins

pytestmark = pytest.mark.gpu

import quantax_amd as qtx  # noqa: E402

LATTICES = [(1, 5, 16), (4, 4, 16), (3, 11, 16), (8, 8, 16), (5, 13, 16), (10, 10, 16), (16, 8, 16), (9, 15, 16),
            (9, 16, 16), (7, 16, 16), (13, 15, 16), (16, 17, 16), (17, 22, 16), (16, 32, 16),
            (3, 5, 32), (8, 8, 32), (6, 13, 32), (8, 16, 32), (9, 16, 32), (16, 16, 32), (15, 18, 32), (20, 20, 32)]


@pytest.mark.parametrize("L0,L1,C", LATTICES)
@pytest.mark.parametrize("prec,tol", [("fp32", 1e-5), ("bf16x3", 1e-4)])
def test_logpsi_classes(L0, L1, C, prec, tol):
    rng = np.random.default_rng(L0 * 40 + L1 + C)
    act, approx = [("tanh", True), ("erf", False), ("relu", "relu")][(L0 + L1) % 3]
    qtx.sites.Grid([L0, L1])
    nb = 1 if L0 * L1 > 300 else 2
    model = qtx.model.ResConv(nb, C, precision=prec, gelu=act, seed=6)
    model.set_params((model.theta.cpu().numpy() + 0.05 * rng.standard_normal(model.nparams)).astype(np.float32))
    s = rand_spins(rng, 2051, L0 * L1)
    sd = torch.from_numpy(s).cuda()
    many = model.logpsi(sd)
    ref = om.resconv_forward(om.ResConvSpec(nb, C, (L0, L1)), model.theta.cpu().numpy().astype(np.float64), s[:6], approx)[1]
    assert max_rel(many[:6].cpu().numpy(), ref) < tol
    # configurations pair up in the head's merge: slices start at an even one
    for a, n in ((0, 1), (0, 7), (2050, 1), (1000, 33)):
        assert torch.equal(model.logpsi(sd[a: a + n]), many[a: a + n]), (a, n)


@pytest.mark.parametrize("L0,L1,C", [(4, 5, 16), (7, 16, 16), (9, 13, 16), (15, 18, 16), (4, 5, 32), (7, 9, 32), (10, 13, 32)])
@pytest.mark.parametrize("prec,tol", [("fp32", 1e-5), ("bf16x3", 1e-4)])
def test_eloc_classes(L0, L1, C, prec, tol):
    """One sample (four waves per configuration) and the same one among many
    (one or two waves): energies equal to the order of the FP64 sum."""
    rng = np.random.default_rng(L0 + 7 * L1)
    N = L0 * L1
    qtx.sites.Grid([L0, L1], Nparticles=(N // 2, N - N // 2))
    model = qtx.model.ResConv(1, C, precision=prec, seed=8)
    H, Ho = qtx.operator.Heisenberg(msr=True), oop.heisenberg([L0, L1], 1.0, 1, True)
    s = rand_spins(rng, 90, N, nup=N // 2)
    sd = torch.from_numpy(s).cuda()
    la = model.logpsi(sd)
    e, nc = model.eloc(H, sd, la)
    theta = model.theta.cpu().numpy().astype(np.float64)
    spec = om.ResConvSpec(1, C, (L0, L1))
    ref = oop.oloc(s[:2], lambda x: om.resconv_forward(spec, theta, x), Ho)
    assert max_rel(e[:2].cpu().numpy(), ref) < tol
    for i in (0, 44, 89):
        e1, n1 = model.eloc(H, sd[i: i + 1], la[i: i + 1])
        assert int(n1[0]) == int(nc[i])
        assert abs(float(e1[0] - e[i])) <= 1e-12 * max(1.0, abs(float(e[i]))) * 4
