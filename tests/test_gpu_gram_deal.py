"""The split-bf16 Gram on both sides of the line where super-blocks are dealt to
the XCDs one by one (96 tile rows of 128), with a ragged last super-row and tile.

Against the float64 product on the GPU.  Tolerance per product: both splits drop
2^-18, lo * lo is left out (2^-18), inputs are rounded to single precision and
sums of 256 columns x 3 products run in it: (3 2^-18 + 770 2^-24) sum |a||b|."""

import pytest
import torch

from quantax_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [12159, 12161, 12300, 13313])
def test_gram_split(n):
    gen = torch.Generator(device="cuda").manual_seed(n)
    np_ = n + 65
    O = torch.randn(n, np_, device="cuda", generator=gen)
    mean = O.mean(0, dtype=torch.float64)
    nws = int(_lib.lib().qtx_gram_ws_bytes(n, np_, 2))
    ws = torch.empty(nws, dtype=torch.uint8, device="cuda")
    T = torch.full((n, n), float("nan"), dtype=torch.float64, device="cuda")
    _lib.call("qtx_gram", _lib.stream(), _lib.QTX_F32, O.data_ptr(), mean.data_ptr(), None, n, np_, 2, T.data_ptr(),
              ws.data_ptr(), nws)
    A = (O.double() - mean) / n**0.5
    bound = (3 * 2.0**-18 + 770 * 2.0**-24) * (A.abs() @ A.abs().T)
    assert torch.equal(T, T.T)
    assert bool(((T - A @ A.T).abs() <= bound).all())
