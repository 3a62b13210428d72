"""The fused ResConv Metropolis kernels run no forward for a proposal that
leaves the spins unchanged, fetch their random words 64 steps at a time and
let the chains of a workgroup run at different steps: spins, amplitudes and
counters against the generic step (propose, forward, accept: every proposal
evaluated, all chains in lock-step) bit for bit, over step counts around the
64-step fetch, odd chain counts and both proposal kinds (needs an MI355X)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

import quantax_amd as qtx  # noqa: E402


@pytest.mark.parametrize("L,C,prec", [(16, 16, "bf16x3"), (16, 16, "fp32"), (10, 16, "fp32"), (6, 16, "bf16x3"),
                                      (20, 32, "bf16x3"), (6, 32, "fp32")])
@pytest.mark.parametrize("kind", ["exchange", "flip"])
def test_fused_equals_generic(L, C, prec, kind):
    N = L * L
    qtx.sites.Square(L, Nparticles=(N // 2, N - N // 2))
    state = qtx.state.Variational(qtx.model.ResConv(2, C, precision=prec, seed=2))
    cls = qtx.sampler.SpinExchange if kind == "exchange" else qtx.sampler.LocalFlip
    ns = 5 if L == 20 else 37
    a = cls(state, ns, thermal_steps=0, seed=9)
    b = cls(state, ns, thermal_steps=0, seed=9)
    b.force_generic = True
    for nsteps in (1, 63, 64, 65, 130) if L < 20 else (1, 65):
        sa, sb = a.sweep(nsteps), b.sweep(nsteps)
        assert torch.equal(sa.spins, sb.spins), nsteps
        assert torch.equal(sa.psi.logabs, sb.psi.logabs), nsteps
        assert torch.equal(a.n_accept, b.n_accept) and torch.equal(a.n_near, b.n_near), nsteps
    assert int(a.n_accept.sum()) > 0


def test_no_movable_spin():
    """All spins equal: every exchange is a null move and the chains stand still."""
    qtx.sites.Square(6, Nparticles=(36, 0))
    state = qtx.state.Variational(qtx.model.ResConv(1, 16, seed=2))
    smp = qtx.sampler.SpinExchange(state, 3, thermal_steps=0, seed=1)
    before = smp._spins.clone()
    la = smp._logabs.clone()
    out = smp.sweep(100)
    assert torch.equal(out.spins, before) and torch.equal(out.psi.logabs, la)
    assert int(smp.n_accept.sum()) == 0 and np.isfinite(la.cpu().numpy()).all()
