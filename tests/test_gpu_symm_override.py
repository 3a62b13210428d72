"""A projected model with a logpsi of its own (a subclass's, or one set on the object)
is evaluated through it, in the state and in the sampler (needs an MI355X)."""
import numpy as np
import pytest
import torch

import quantax_amd as qtx

pytestmark = pytest.mark.gpu


def _extra(s):
    return 0.3 * (s[:, 0] * s[:, 1]).to(torch.float64)


class Jastrowed(qtx.model.RBM_Dense):
    def logpsi(self, s, h_out=False):
        return super().logpsi(s) + _extra(s)


@pytest.mark.parametrize("how", ["subclass", "object"])
def test_own_logpsi(how):
    qtx.sites.Square(4, Nparticles=(8, 8))
    kw = dict(dtype=np.float64, init_std=0.1, seed=3)
    if how == "subclass":
        model = Jastrowed(12, **kw)
    else:
        model = qtx.model.RBM_Dense(12, **kw)
        plain = model.logpsi
        model.logpsi = lambda s, h_out=False: plain(s) + _extra(s)
    symm = qtx.symmetry.C4v()
    state = qtx.state.Variational(model, symm=symm)
    rng = np.random.default_rng(0)
    s = torch.as_tensor(np.stack([rng.permutation([1, -1] * 8) for _ in range(9)]).astype(np.int8), device="cuda")
    sg, la = symm.project(model.logpsi(symm.images(s)))
    psi = state(s)
    assert torch.equal(psi.logabs, la) and torch.equal(psi.sign, sg)
    smp = qtx.sampler.SpinExchange(state, 9, initial_spins=s, thermal_steps=0, seed=1)
    out = smp.sweep(20)
    assert torch.equal(out.psi.logabs, state(out.spins).logabs)


class Scaled(qtx.state.Variational):
    """psi^2: other acceptances than psi."""

    def __call__(self, s):
        psi = super().__call__(s)
        return qtx.utils.LogArray(psi.sign, 2 * psi.logabs)


class NoInversion(qtx.symmetry.Symmetry):
    def project(self, logabs, weights=False):
        assert not weights
        half = logabs.reshape(-1, self.nsymm)[:, : self.nsymm // 2]
        la = torch.logsumexp(half, 1)
        return torch.ones_like(la), la


@pytest.mark.parametrize("how", ["state", "symmetry"])
def test_own_amplitudes_and_projection(how):
    qtx.sites.Square(4, Nparticles=(8, 8))
    model = qtx.model.RBM_Dense(12, dtype=np.float64, init_std=0.1, seed=3)
    symm = qtx.symmetry.C4v() if how == "state" else NoInversion(Z2_inversion=1)
    state = (Scaled if how == "state" else qtx.state.Variational)(model, symm=symm)
    rng = np.random.default_rng(0)
    s = torch.as_tensor(np.stack([rng.permutation([1, -1] * 8) for _ in range(9)]).astype(np.int8), device="cuda")
    sg, la = symm.project(model.logpsi(symm.images(s)))
    assert torch.equal(state(s).logabs, 2 * la if how == "state" else la)
    smp = qtx.sampler.SpinExchange(state, 9, initial_spins=s, thermal_steps=0, seed=1)
    out = smp.sweep(20)
    assert torch.equal(out.psi.logabs, state(out.spins).logabs)


def test_the_class_itself_is_fused():
    qtx.sites.Square(4, Nparticles=(8, 8))
    model = qtx.model.RBM_Dense(12, dtype=np.float64, init_std=0.1)
    assert qtx.state.Variational(model, symm=qtx.symmetry.C4v()).fused_symm
