"""Any-lattice ResConv forwards around the numbers of configurations where the
waves per configuration change: a configuration's amplitude has the same bits
in a batch of any size."""

import numpy as np
import pytest
import torch

import quantax_amd as qtx

pytestmark = pytest.mark.gpu

LINES = (511, 512, 768, 769, 1024, 1025, 1536, 1537, 1792, 1793)


@pytest.mark.parametrize("L0,L1", [(4, 4), (5, 6), (7, 8), (9, 12), (12, 12)])
@pytest.mark.parametrize("C,prec", [(16, "fp32"), (16, "bf16x3"), (32, "fp32"), (32, "bf16x3")])
def test_amplitudes_do_not_depend_on_the_batch(L0, L1, C, prec):
    qtx.sites.Grid([L0, L1])
    model = qtx.model.ResConv(2, C, precision=prec)
    rng = np.random.default_rng(L0 * L1 + C)
    s = torch.as_tensor(rng.choice([-1, 1], (max(LINES), L0 * L1)).astype(np.int8), device="cuda")
    ref = torch.cat([model.logpsi(s[i:i + 100]) for i in range(0, len(s), 100)])
    for ns in LINES:
        assert torch.equal(model.logpsi(s[:ns]), ref[:ns]), ns
