"""The packed image of a ResConv: everything that a forward, a sweep's or the
Jacobian's kernel reads is written by the pack (over an image of NaNs), and nothing
else is kept or written."""
import numpy as np
import pytest
import torch

import quantax_amd as qtx
from quantax_amd import _lib

CASES = [(6, 6, 16), (16, 16, 16), (5, 7, 32), (18, 18, 32)]


@pytest.mark.parametrize("L0,L1,C", CASES)
@pytest.mark.parametrize("nb", [1, 3])
def test_fp32_images_hold_their_weights_once(L0, L1, C, nb):
    """Both directions' fragments, the copy of theta and the biases, and the window
    kernel's own fragments on 16 x 16 with 16 channels; rounding up to 256 bytes."""
    d = _lib.QtxResConvDesc()
    d.nblocks, d.channels, d.L0, d.L1 = nb, C, L0, L1
    d.precision, d.activation = _lib.QTX_CONV_FP32, _lib.QTX_ACT_GELU_TANH
    n = _lib.lib().qtx_resconv_nparams(d) + 10 * C + 2 * nb * C + 2 * 2 * nb * 9 * C * C
    if (L0, L1, C) == (16, 16, 16):
        n += 2 * nb * 9 * C * C
    assert 4 * n <= _lib.lib().qtx_resconv_packed_bytes(d) < 4 * n + 5 * 256


@pytest.mark.gpu
@pytest.mark.parametrize("L0,L1,C", CASES)
@pytest.mark.parametrize("prec", ["fp32", "bf16x3"])
@pytest.mark.parametrize("nb", [1, 3])
def test_pack_writes_what_is_read(L0, L1, C, prec, nb):
    qtx.sites.Grid([L0, L1])
    model = qtx.model.ResConv(nb, C, precision=prec, seed=1)
    rng = np.random.default_rng(0)
    s = torch.as_tensor(rng.choice([-1, 1], (9, L0 * L1)).astype(np.int8), device="cuda")
    la, O = model.logpsi(s), model.jacobian(s)
    model.packed.fill_(255)  # NaNs in float32 and bfloat16
    model.repack()
    assert torch.isfinite(la).all() and torch.isfinite(O).all()
    assert torch.equal(model.logpsi(s), la) and torch.equal(model.jacobian(s), O)
