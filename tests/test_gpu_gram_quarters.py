"""The FP64 / FP32 Gram on both sides of its deal of 64 x 64 tiles and 32 x 32
quarters over the XCDs: less than a round of tiles (all quarters), whole rounds,
whole rounds and up to 16 tiles more, 17 and more; row counts that end inside a
tile, a quarter and a 16-row block; np that is no multiple of a column chunk.

Against the float64 product.  Tolerance from the forms of the sums: FP64 (np +
8) 2^-53 sum |a||b|; FP32 inputs rounded to 2^-24 and sums of at most 256 terms
in single precision: (256 + 4) 2^-24 sum |a||b|."""

import numpy as np
import pytest
import torch

from quantax_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 97, 300, 700, 1000, 1100, 1400, 1450, 1984, 2048])
@pytest.mark.parametrize("more,weights", [(50, False), (273, True)])
@pytest.mark.parametrize("gram", ["fp64", "fp32"])
def test_gram(n, more, weights, gram):
    np_ = n + more  # the sample-space product
    rng = np.random.default_rng(n + np_)
    O = rng.standard_normal((n, np_)).astype(np.float32)
    mean = rng.standard_normal(np_) * 0.1
    r = rng.random(n) + 0.5
    A = (O.astype(np.float64) - mean) * np.sqrt((r if weights else np.ones(n)) / n)[:, None]
    g = {"fp64": 0, "fp32": 1}[gram]
    Od, md, rd = (torch.as_tensor(v, device="cuda") for v in (O, mean, r))
    T = torch.full((n, n), float("nan"), dtype=torch.float64, device="cuda")
    _lib.call("qtx_gram", _lib.stream(), _lib.QTX_F32, Od.data_ptr(), md.data_ptr(), rd.data_ptr() if weights else None,
              n, np_, g, T.data_ptr(), None, 0)
    T = T.cpu().numpy()
    assert np.array_equal(T, T.T)
    bound = np.abs(A) @ np.abs(A).T * ((np_ + 8) * 2.0**-53 if g == 0 else 260 * 2.0**-24)
    assert np.all(np.abs(T - A @ A.T) <= bound)
