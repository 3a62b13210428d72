"""The ResConv Jacobian at the edges of its kernel's tiles and loops against
the oracle (needs an MI355X): lattices of one ragged tile up to the largest
accepted, every tiles-per-wave class (NT <= 4, 8, 16, 32 tiles of 16 sites),
one block (no input gradient), sample counts around the number of workgroup
slots, and O rows that are not 16-byte aligned.  FP32 products and sums: 1e-5
of the largest entry, as for the other FP32 network paths."""
import numpy as np
import pytest
import torch

from oracle import models as om
from tests.helpers import rand_spins

pytestmark = pytest.mark.gpu

import quantax_amd as qtx  # noqa: E402
from quantax_amd import _lib  # noqa: E402


@pytest.mark.parametrize("L0,L1,C,nb", [(3, 5, 16, 1), (2, 8, 16, 2), (8, 8, 16, 2), (5, 13, 16, 2), (9, 14, 16, 2),
                                        (1, 16, 16, 2), (13, 20, 16, 2), (16, 32, 16, 1), (3, 4, 32, 1), (9, 7, 32, 2),
                                        (11, 12, 32, 2), (20, 20, 32, 1)])
@pytest.mark.parametrize("act", ["tanh", "erf", "relu"])
def test_jacobian_tile_edges(L0, L1, C, nb, act):
    if act != "tanh" and L0 * L1 > 130:
        pytest.skip("activations are covered by the smaller lattices")
    rng = np.random.default_rng(L0 * 100 + L1)
    qtx.sites.Grid([L0, L1])
    model = qtx.model.ResConv(nb, C, precision="bf16x3" if nb == 2 else "fp32", gelu=act, seed=4)
    th = model.theta.cpu().numpy().astype(np.float64) + 0.05 * rng.standard_normal(model.nparams)
    model.set_params(th.astype(np.float32))
    theta = model.theta.cpu().numpy().astype(np.float64)
    ns = 5
    s = rand_spins(rng, ns, L0 * L1)
    sd = torch.from_numpy(s).cuda()
    spec = om.ResConvSpec(nb, C, (L0, L1))
    kw = {} if act == "tanh" else {"approximate": False if act == "erf" else "relu"}
    ref = om.resconv_jacobian(spec, theta, s, **kw)
    tol = 1e-5 * max(1.0, np.abs(ref).max())
    assert np.max(np.abs(model.jacobian(sd).cpu().numpy() - ref)) < tol
    # O one float past a 16-byte boundary
    buf = torch.full((ns * model.nparams + 1,), float("nan"), dtype=torch.float32, device="cuda")
    nws = int(_lib.lib().qtx_resconv_jacobian_ws_bytes(model.desc, ns))
    ws = torch.empty(nws, dtype=torch.uint8, device="cuda")
    _lib.call("qtx_resconv_jacobian", _lib.stream(), model.desc, model.packed.data_ptr(), sd.data_ptr(), ns,
              buf[1:].data_ptr(), ws.data_ptr(), nws)
    assert np.max(np.abs(buf[1:].view(ns, -1).cpu().numpy() - ref)) < tol


def test_more_samples_than_slots():
    """Workgroups loop over samples beyond 768: every row equals the row of a
    launch of that sample alone (the same kernel and order: bit for bit)."""
    rng = np.random.default_rng(3)
    qtx.sites.Square(4)
    model = qtx.model.ResConv(2, 16, seed=1)
    sd = torch.from_numpy(rand_spins(rng, 1700, 16)).cuda()
    O = model.jacobian(sd)
    for n in (0, 767, 768, 1535, 1536, 1699):
        assert torch.equal(O[n], model.jacobian(sd[n: n + 1])[0])
