"""ResConv sweeps with enough chains for one or two waves per chain: the instances of
the Metropolis kernel that only large launches take (from 512 chains on a single tile,
1537 up to four tiles and 1537 / 1793 beyond), whose chains end and break out one by
one (one wave) or share barriers at different steps (two).

Spins, amplitudes and counters against the generic step (propose, forward, accept) bit
for bit, at odd chain counts on both sides of each line and step counts around the
64-step fetch."""
import pytest
import torch

import quantax_amd as qtx

pytestmark = pytest.mark.gpu

# sites: 16 (a single tile), 30 and 56 (up to four, ragged), 100 (seven), 130 (nine, ragged)
CASES = [(4, 4, (511, 513)), (5, 6, (1535, 1537)), (7, 8, (1537,)), (10, 10, (1537, 1793)), (10, 13, (1791, 1793))]


@pytest.mark.parametrize("L0,L1,chains", CASES)
@pytest.mark.parametrize("C,prec", [(16, "fp32"), (16, "bf16x3"), (32, "fp32"), (32, "bf16x3")])
@pytest.mark.parametrize("kind", ["exchange", "flip"])
def test_fused_equals_generic(L0, L1, chains, C, prec, kind):
    N = L0 * L1
    qtx.sites.Grid([L0, L1], Nparticles=(N // 2, N - N // 2))
    state = qtx.state.Variational(qtx.model.ResConv(1, C, precision=prec, seed=2))
    cls = qtx.sampler.SpinExchange if kind == "exchange" else qtx.sampler.LocalFlip
    for ns in chains:
        a = cls(state, ns, thermal_steps=0, seed=9)
        b = cls(state, ns, thermal_steps=0, seed=9)
        b.force_generic = True
        for nsteps in (1, 65):
            sa, sb = a.sweep(nsteps), b.sweep(nsteps)
            assert torch.equal(sa.spins, sb.spins), (ns, nsteps)
            assert torch.equal(sa.psi.logabs, sb.psi.logabs), (ns, nsteps)
            assert torch.equal(a.n_accept, b.n_accept) and torch.equal(a.n_near, b.n_near), (ns, nsteps)
        assert int(a.n_accept.sum()) > 0


def test_chains_that_cannot_move_beside_ones_that_can():
    """Two chains share a workgroup (9 to 16 tiles): every other one has all spins
    equal, no exchange to make, and waits for its neighbour."""
    qtx.sites.Grid([10, 13], Nparticles=(65, 65))
    state = qtx.state.Variational(qtx.model.ResConv(1, 16, seed=2))
    s = torch.ones((1793, 130), dtype=torch.int8)
    s[1::2, ::2] = -1
    a = qtx.sampler.SpinExchange(state, 1793, initial_spins=s, thermal_steps=0, seed=4)
    b = qtx.sampler.SpinExchange(state, 1793, initial_spins=s, thermal_steps=0, seed=4)
    b.force_generic = True
    x, y = a.sweep(65), b.sweep(65)
    assert torch.equal(x.spins, y.spins) and torch.equal(x.psi.logabs, y.psi.logabs)
    assert torch.equal(x.spins[::2].cpu(), s[::2]) and torch.equal(a.n_accept, b.n_accept)
