"""RBM sampling and local energies in windows of 64 steps / candidates: around
the windows' ends, at lattice sizes around 64 sites and hidden units around the
registers' limits, against the general path (propose, full forward, accept) and
the sum over listed connected configurations.

In float64 the two paths' log psi agree to ~1e-13, so every decision and every
counter is the same; the energies are sums of at most noff terms of relative
error a few 1e-13 each, far below 1e-10 of their magnitudes' sum."""

import numpy as np
import pytest
import torch

import quantax_amd as qtx

pytestmark = pytest.mark.gpu

CONVENTION = {"heisenberg": 1.0, "ising": 1.0}  # both operators in sigma matrices


def _state(L, M, seed, nup):
    qtx.sites.Chain(L, Nparticles=None if nup is None else (nup, L - nup))
    model = qtx.model.RBM_Dense(M, dtype=np.float64, init_std=0.15, seed=seed)
    return qtx.state.Variational(model)


@pytest.mark.parametrize("L,M,nup", [(2, 1, 1), (7, 5, 3), (64, 64, 32), (65, 63, 30), (66, 130, 1), (130, 257, 64),
                                     (20, 513, 10), (12, 6, 12), (9, 65, None), (70, 200, None)])
@pytest.mark.parametrize("steps", [1, 63, 64, 65, 130])
def test_sweep_matches_general_path(L, M, nup, steps):
    state = _state(L, M, 3, nup)
    kind = qtx.sampler.LocalFlip if nup is None else qtx.sampler.SpinExchange
    out = []
    for generic in (False, True):
        smp = kind(state, 33, thermal_steps=0, sweep_steps=steps, seed=5)
        smp.force_generic = generic
        s = smp.sweep()
        out.append((s.spins.clone(), smp.n_accept.clone(), s.psi.logabs.clone()))
    assert torch.equal(out[0][0], out[1][0])
    assert torch.equal(out[0][1], out[1][1])
    assert torch.allclose(out[0][2], out[1][2], rtol=1e-11, atol=1e-11)


@pytest.mark.parametrize("L,M", [(4, 3), (63, 17), (64, 65), (65, 400), (130, 9), (9, 600)])
@pytest.mark.parametrize("model", ["heisenberg", "ising"])
def test_eloc_matches_connected_sum(L, M, model):
    state = _state(L, M, 7, None if model == "ising" else L // 2)
    H = qtx.operator.Ising(h=0.7) if model == "ising" else qtx.operator.Heisenberg()
    spins = (qtx.sampler.LocalFlip if model == "ising" else qtx.sampler.SpinExchange)(
        state, 21, thermal_steps=8, seed=2).sweep().spins
    eloc = H.Oloc(state, qtx.sampler.Samples(spins, state(spins), None, None)).cpu().numpy()
    W = state.model.theta.double().cpu().numpy()
    s = spins.cpu().numpy().astype(np.float64)
    Wm, b = W[: M * L].reshape(M, L), W[M * L:]
    lpsi = lambda x: np.log(np.cosh(x @ Wm.T + b)).sum(-1)
    ref = np.zeros(len(s))
    for i in range(L):
        j = (i + 1) % L
        if L == 2 and i == 1:
            continue
        zz = s[:, i] * s[:, j]
        if model == "ising":
            t = s.copy()
            t[:, i] *= -1
            ref += -zz - 0.7 * np.exp(lpsi(t) - lpsi(s))
        else:
            t = s.copy()
            t[:, [i, j]] = t[:, [j, i]]
            ref += zz + np.where(zz < 0, 2 * np.exp(lpsi(t) - lpsi(s)), 0.0)
    scale = max(1.0, np.abs(ref).max())
    assert np.abs(eloc - CONVENTION[model] * ref).max() <= 1e-10 * scale, (eloc[:4], ref[:4])
