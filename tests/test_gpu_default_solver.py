"""The optimiser as it comes, SR(state, H) with its default solver (a cutoff of
1e-12), on the samples of a sweep: their reweighting factors are ones, so the
solve takes the small-cutoff route that deflates the null direction 1, as it does
without factors.  Any other factors have another null direction: dsyevd."""
import numpy as np
import pytest
import torch

import quantax_amd as qtx

pytestmark = pytest.mark.gpu


def _state(ns, reweight=2.0):
    qtx.sites.Chain(10)
    H = qtx.operator.Ising(h=1.0)
    state = qtx.state.Variational(qtx.model.RBM_Dense(60, dtype=np.float64, init_std=0.3, seed=1))
    return H, state, qtx.sampler.LocalFlip(state, ns, reweight=reweight, thermal_steps=40, seed=2).sweep()


def _tol(O):
    """Both solves are accepted with a normwise backward error of 1e-15; the
    products around them add the usual (ns + np) u.  Times the condition number of
    the deflated T on its range."""
    ns, np_ = O.shape
    A = (O - O.mean(0)) / np.sqrt(ns)
    lam = np.linalg.eigvalsh(A @ A.T)
    lam = lam[lam > 1e-11 * lam[-1]]
    return 32 * (ns + np_) * 2.0**-53 * lam[-1] / lam[0]


@pytest.mark.parametrize("ns", [24, 40])
@pytest.mark.parametrize("opt", ["SR", "SPRING", "MARCH", "AdamSR"])
def test_sweep_samples_take_the_route_without_factors(ns, opt):
    H, state, _ = _state(ns)
    g = np.random.default_rng(ns)
    # distinct configurations: T is regular but for its null direction
    bits = g.permutation(1024)[:ns]
    spins = torch.as_tensor(np.where(bits[:, None] >> np.arange(10) & 1, 1, -1).astype(np.int8), device="cuda")
    psi = state(spins)
    one = qtx.sampler.LocalFlip(state, ns, thermal_steps=0, seed=3)._reweight_factor(psi.logabs)
    out = []
    for r in (None, one):
        o = getattr(qtx.optimizer, opt)(state, H)
        step = o.get_step(qtx.sampler.Samples(spins, psi, None, r))
        out.append((step.cpu().numpy(), qtx.optimizer.last_solve_info()))
    assert out[0][1]["path"] == out[1][1]["path"] == "shifted_cholesky"
    assert out[1][1]["fallback"] is None
    tol = _tol(state.jacobian(spins).double().cpu().numpy())
    if opt == "SR":
        assert np.linalg.norm(out[1][0] - out[0][0]) <= tol * np.linalg.norm(out[0][0])


@pytest.mark.parametrize("solver", ["shift", "pinv"])
@pytest.mark.parametrize("form", ["device", "single", "one", "strided", "host"])
def test_ones_give_the_step_without_factors(solver, form):
    """In whatever form; solvers whose route does not look at the factors."""
    H, state, smp = _state(40)
    one = torch.ones(40, dtype=torch.float64, device="cuda")
    r = {"device": one, "single": one.float(), "one": one[:1], "strided": one[:1].expand(40), "host": one.cpu()}[form]
    sv = qtx.optimizer.auto_shift_eig(rshift=1e-2, ashift=0.0) if solver == "shift" else qtx.optimizer.auto_pinv_eig(1e-2)
    steps = [qtx.optimizer.SR(state, H, solver=sv).get_step(qtx.sampler.Samples(smp.spins, smp.psi, None, f))
             for f in (None, r)]
    # a condition number of at most 1e2 (40 rows of trace 1 at most, or the cutoff's)
    tol = 32 * (40 + state.nparams) * 2.0**-53 * 1e2 * float(steps[0].norm())
    assert float((steps[1] - steps[0]).norm()) <= tol


def test_other_factors_take_dsyevd():
    H, state, smp = _state(40, reweight=1.5)
    assert not bool((smp.reweight_factor == 1.0).all())
    qtx.optimizer.SR(state, H).get_step(smp)
    info = qtx.optimizer.last_solve_info()
    assert info["path"] == "syevd" and info["fallback"] == "small_cutoff"


@pytest.mark.parametrize("at", [0, 63, 1023, 1024, 1499])
def test_one_other_factor_is_seen(at):
    """Wherever it stands among 1500."""
    rng = np.random.default_rng(at)
    O = torch.as_tensor(rng.standard_normal((1500, 1600)), device="cuda")
    e = torch.as_tensor(rng.standard_normal(1500), device="cuda")
    r = torch.ones(1500, dtype=torch.float64, device="cuda")
    r[at] = 1.0 + 2.0**-52
    qtx.optimizer.solve_step(O, O.mean(0), e - e.mean(), qtx.optimizer.auto_pinv_eig(), r)
    assert qtx.optimizer.last_solve_info()["path"] == "syevd"
