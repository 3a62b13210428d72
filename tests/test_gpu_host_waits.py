"""Sampling and the SR step without the host's looks at device values: the drift
count against the torch expression it replaces (chunk edges, NaN, infinities),
and weights of one giving the same bits as no weights."""

import numpy as np
import pytest
import torch

import quantax_amd as qtx
from quantax_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns", [1, 63, 64, 65, 255, 256, 257, 1000])
def test_drift_count(ns):
    rng = np.random.default_rng(ns)
    a = rng.normal(0.0, 30.0, ns)
    b = a + np.where(rng.random(ns) < 0.4, rng.choice([0.1, -0.02, 1e-5, 1e-12], ns), 0.0)
    b[rng.random(ns) < 0.1] = np.nan
    b[rng.random(ns) < 0.1] = -np.inf
    a[rng.random(ns) < 0.1] = -np.inf
    a, b = torch.as_tensor(a, device="cuda"), torch.as_tensor(b, device="cuda")
    count = torch.full((1,), 77, dtype=torch.int32, device="cuda")
    _lib.call("qtx_drift_count", _lib.stream(), a.data_ptr(), b.data_ptr(), ns, count.data_ptr())
    close = (torch.abs(torch.exp(a) - torch.exp(b)) < 1e-8) | (torch.abs(torch.exp(a - b) - 1) < 1e-3)
    assert int(count.item()) == int((~close).sum().item())


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_weights_of_one(dtype):
    """The same step whether the factors are absent, ones in the kernels' layout,
    or ones that the kernels cannot read (a strided view, single precision)."""
    qtx.sites.Chain(8)
    H = qtx.operator.Ising(h=1.0)
    state = qtx.state.Variational(qtx.model.RBM_Dense(8, dtype=dtype, init_std=0.05, seed=1))
    spins = qtx.sampler.LocalFlip(state, 60, thermal_steps=4, seed=2).sweep().spins
    psi = state(spins)
    one = torch.ones(60, dtype=torch.float64, device="cuda")
    out = []
    for r in (None, one, one[:1].expand(60), one.float(), one[:1]):
        opt = qtx.optimizer.SR(state, H, solver=qtx.optimizer.auto_shift_eig(rshift=0.0, ashift=1e-3))
        ebar = opt.get_Ebar(qtx.sampler.Samples(spins, psi, None, r))
        out.append((ebar, opt.energy, opt.VarE))
        assert torch.isfinite(opt.get_step(qtx.sampler.Samples(spins, psi, None, r))).all()
    for e, en, var in out[1:]:
        assert torch.equal(e, out[0][0]) and en == out[0][1] and var == out[0][2]
