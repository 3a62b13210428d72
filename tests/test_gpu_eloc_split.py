"""E_loc with a sample's candidates split over several workgroups against the
unsplit launch (needs an MI355X): the same forwards, so the energies agree to
the order of an FP64 sum of at most 1600 terms (1600 x 2^-53 = 1.8e-13 of the
sum of their moduli) and the candidate counts exactly."""
import numpy as np
import pytest
import torch

from tests.helpers import rand_spins

pytestmark = pytest.mark.gpu

import quantax_amd as qtx  # noqa: E402
from quantax_amd import _lib  # noqa: E402


@pytest.mark.parametrize("L,C,prec,ham", [(16, 16, "bf16x3", "j1j2"), (10, 16, "fp32", "j1j2"), (20, 32, "bf16x3", "j1j2"),
                                          (6, 32, "fp32", "ising"), (4, 16, "bf16x3", "j1j2")])
@pytest.mark.parametrize("ns", [1, 37, 700])
def test_split_equals_unsplit(L, C, prec, ham, ns):
    if L == 20 and ns > 37:
        pytest.skip("covered by the smaller lattices")
    N = L * L
    nup = N // 2 if ham == "j1j2" else None
    qtx.sites.Square(L, Nparticles=(N // 2, N - N // 2))
    model = qtx.model.ResConv(2, C, precision=prec, seed=5)
    H = (qtx.operator.Heisenberg(J=[1, 0.5], n_neighbor=[1, 2], msr=True) if ham == "j1j2"
         else qtx.operator.Ising(h=0.7, J=1.3))
    s = rand_spins(np.random.default_rng(L + ns), ns, N, nup=nup)
    s[0] = 1  # no antiparallel bond: an empty candidate list under J1-J2
    sd = torch.from_numpy(s).cuda()
    la = model.logpsi(sd)
    e, nc = model.eloc(H, sd, la)
    ref = torch.empty_like(e)
    ncr = torch.empty_like(nc)
    _lib.call("qtx_resconv_eloc", _lib.stream(), model.desc, model.packed.data_ptr(), H.device_tables(), sd.data_ptr(),
              la.data_ptr(), ns, ref.data_ptr(), ncr.data_ptr())
    assert torch.equal(nc, ncr)
    assert torch.all((e - ref).abs() <= 1e-12 * ref.abs().clamp(min=1.0) * 4)
