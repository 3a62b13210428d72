"""FP32 forwards of 16 channels around the numbers of configurations from which two, five
and six tiles take one wave, nine and more two: a configuration's amplitude has the same
bits in a batch of any size.  Lattices one and two sites wide (the source table's wraps)
against the oracle, tolerance of the FP32 ResConv tests."""
import numpy as np
import pytest
import torch

import quantax_amd as qtx
from oracle import models as om
from tests.helpers import max_rel

pytestmark = pytest.mark.gpu


def _batch(L0, L1, ns):
    qtx.sites.Grid([L0, L1])
    rng = np.random.default_rng(L0 * L1)
    return (qtx.model.ResConv(2, 16, seed=6),
            torch.as_tensor(rng.choice([-1, 1], (ns, L0 * L1)).astype(np.int8), device="cuda"))


@pytest.mark.parametrize("L0,L1", [(3, 6), (2, 16), (5, 13), (6, 16), (8, 10), (10, 13), (8, 17), (10, 16), (16, 15)])
def test_amplitudes_do_not_depend_on_the_batch(L0, L1):
    model, s = _batch(L0, L1, 1281)
    ref = torch.cat([model.logpsi(s[i:i + 100]) for i in range(0, len(s), 100)])
    for ns in (768, 769, 1024, 1025, 1280, 1281):
        assert torch.equal(model.logpsi(s[:ns]), ref[:ns]), ns


@pytest.mark.parametrize("L0,L1", [(1, 1), (1, 7), (7, 1), (2, 9), (18, 2), (1, 300), (300, 1), (2, 2)])
def test_narrow_lattices(L0, L1):
    model, s = _batch(L0, L1, 6)
    ref = om.resconv_forward(om.ResConvSpec(2, 16, (L0, L1)), model.theta.cpu().numpy().astype(np.float64),
                             s.cpu().numpy(), True)[1]
    assert max_rel(model.logpsi(s).cpu().numpy(), ref) < 1e-5
