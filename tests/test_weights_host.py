"""The reweighting factors that an SR step hands to its kernels: never a tensor
that lives on the host or has another layout than the kernels read."""
import numpy as np
import pytest
import torch

import quantax_amd as qtx
from quantax_amd.optimizer import QNGD

SPINS = np.ones((5, 4), np.int8)


@pytest.mark.parametrize("spins", [SPINS, torch.from_numpy(SPINS)])
@pytest.mark.parametrize("r", [None, torch.ones(5, dtype=torch.float64), torch.ones(5), np.ones(5),
                               torch.ones(1, dtype=torch.float64).expand(5), torch.ones(1, dtype=torch.float64)])
def test_host_ones_need_no_kernel(spins, r):
    assert QNGD._weights(qtx.sampler.Samples(spins, None, None, r)) is None


def test_one_factor_per_sample():
    with pytest.raises(ValueError, match="one reweighting factor"):
        QNGD._weights(qtx.sampler.Samples(SPINS, None, None, torch.tensor([1.0, 2.0])))


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["host", "single", "strided", "numpy"])
def test_other_layouts_are_copied(form):
    """Factors of two and a half in any form: the step of the float64 device tensor,
    up to the order of its sums (16 (ns + np) u cond, cond below 10 with this shift)."""
    qtx.sites.Chain(8)
    H = qtx.operator.Ising(h=1.0)
    state = qtx.state.Variational(qtx.model.RBM_Dense(8, dtype=np.float64, init_std=0.05, seed=1))
    spins = qtx.sampler.LocalFlip(state, 60, thermal_steps=4, seed=2).sweep().spins
    psi = state(spins)
    base = torch.tensor([0.5, 2.0] * 30, dtype=torch.float64, device="cuda")
    r = {"host": base.cpu(), "single": base.float(), "strided": base.repeat_interleave(2)[::2],
         "numpy": base.cpu().numpy()}[form]
    out = []
    for f in (base, r):
        opt = qtx.optimizer.SR(state, H, solver=qtx.optimizer.auto_shift_eig(rshift=1.0, ashift=0.0))
        out.append((opt.get_step(qtx.sampler.Samples(spins, psi, None, f)), opt.energy))
    assert out[0][1] == out[1][1]
    assert float((out[0][0] - out[1][0]).norm()) <= 16 * (60 + 72) * 2.0**-53 * 10 * float(out[0][0].norm())
