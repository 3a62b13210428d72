"""The projected float64 RBM without images against the general path (images
-> forward -> projection; propose -> that -> accept) over the kernels'
classes: hidden units and sites at the 16-unit and 4-site edges, groups of one
ragged tile of permutations up to 512 with and without spin inversion (needs
an MI355X).  Both are float64 sums of at most 64 units and 1024 images:
amplitudes to 1e-12 (vanishing ones, below 1e-10 of the largest image, as
such), chains and counters exactly."""
import numpy as np
import pytest
import torch

from tests.helpers import max_rel, rand_spins

pytestmark = pytest.mark.gpu

import quantax_amd as qtx  # noqa: E402

S = qtx.symmetry
GROUPS = {
    "flip": lambda: S.Flip(axis=1, sector=1),
    "z2": lambda: S.SpinInverse(-1),
    "c4v_z2": lambda: S.C4v() @ S.SpinInverse(1),
    "trans_c4v": lambda: S.TransND() @ S.C4v(),
    "all": lambda: S.TransND() @ S.C4v() @ S.SpinInverse(1),
    "c4v_b2_zm": lambda: S.C4v(repr="B2") @ S.SpinInverse(-1),
}


@pytest.mark.parametrize("L,M", [(2, 1), (3, 16), (4, 17), (4, 32), (5, 33), (6, 36), (6, 48), (6, 64), (7, 5), (8, 20), (8, 64)])
@pytest.mark.parametrize("group", list(GROUPS))
def test_fused_equals_general(L, M, group):
    N = L * L
    rng = np.random.default_rng(L * 100 + M)
    qtx.sites.Square(L, Nparticles=(N // 2, N - N // 2))
    model = qtx.model.RBM_Dense(M, dtype=np.float64, init_std=0.3 / np.sqrt(M), seed=M)
    symm = GROUPS[group]()
    state = qtx.state.Variational(model, symm=symm)
    assert state.fused_symm
    s = rand_spins(rng, 33, N, nup=N // 2)
    sd = torch.from_numpy(s).cuda()
    psi = state(sd)
    img = model.logpsi(symm.images(sd))
    sg, la = symm.project(img)
    big = img.view(33, -1).max(1).values.cpu().numpy()
    ref, got = la.cpu().numpy(), psi.logabs.cpu().numpy()
    zero = ~np.isfinite(ref) | (ref - big < np.log(1e-10))
    assert np.array_equal(zero, ~np.isfinite(got) | (got - big < np.log(1e-10)))
    ok = ~zero
    # a sum that cancels to a fraction f of its largest term keeps 1e-13 / f
    lost = np.exp(big[ok] - ref[ok])
    assert np.all(np.abs(got[ok] - ref[ok]) <= 1e-12 * np.maximum(1.0, np.abs(ref[ok])) + 1e-13 * lost)
    assert np.array_equal(psi.sign.cpu().numpy()[ok], sg.cpu().numpy()[ok])
    if zero.any():
        return  # accept / reject on round-off amplitudes
    for cls in (qtx.sampler.SpinExchange, qtx.sampler.LocalFlip):
        if cls is qtx.sampler.LocalFlip and group in ("z2", "c4v_b2_zm", "flip"):
            continue  # leaves the sector, where amplitudes may vanish
        a = cls(state, 5, thermal_steps=0, initial_spins=sd[:5], seed=3)
        b = cls(state, 5, thermal_steps=0, initial_spins=sd[:5], seed=3)
        b.force_generic = True
        for n in (1, 65):
            x, y = a.sweep(n), b.sweep(n)
            assert torch.equal(x.spins, y.spins) and torch.equal(x.psi.sign, y.psi.sign)
            assert max_rel(x.psi.logabs.cpu().numpy(), y.psi.logabs.cpu().numpy()) < 1e-11
            assert torch.equal(a.n_accept, b.n_accept) and torch.equal(a.n_near, b.n_near)


def test_general_path_beyond_the_limits():
    """More hidden units than the fragments hold, and float32: the general path."""
    qtx.sites.Square(4, Nparticles=(8, 8))
    symm = S.C4v()
    assert not qtx.state.Variational(qtx.model.RBM_Dense(65, dtype=np.float64, init_std=0.1), symm=symm).fused_symm
    assert not qtx.state.Variational(qtx.model.RBM_Dense(16, dtype=np.float32, init_std=0.1), symm=symm).fused_symm
