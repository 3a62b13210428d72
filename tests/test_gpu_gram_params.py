"""S = Obar^T Obar of the SR branch (ns >= np) at the edges of its split: 16
columns per tile, groups of four samples dealt to 16 waves, 256 samples per part.

Against the float64 product.  Tolerance: a sum of ns products in any order, each
with three roundings: (ns + 8) 2^-53 sum |a||b|."""

import numpy as np
import pytest
import torch

import quantax_amd as qtx
from oracle import sr as osr
from quantax_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns,np_", [(1, 1), (3, 2), (15, 15), (16, 16), (17, 17), (64, 5), (255, 31), (256, 32),
                                    (257, 33), (511, 64), (513, 65), (1024, 272), (1025, 100), (3000, 530)])
@pytest.mark.parametrize("dtype,weights", [(np.float32, False), (np.float64, True)])
def test_gram(ns, np_, dtype, weights):
    rng = np.random.default_rng(ns + np_)
    O = rng.standard_normal((ns, np_)).astype(dtype)
    mean = rng.standard_normal(np_) * 0.1
    r = rng.random(ns) + 0.5
    A = (O.astype(np.float64) - mean) * np.sqrt((r if weights else np.ones(ns)) / ns)[:, None]
    Od, md, rd = (torch.as_tensor(v, device="cuda") for v in (O, mean, r))
    S = torch.full((np_, np_), float("nan"), dtype=torch.float64, device="cuda")
    _lib.call("qtx_gram", _lib.stream(), _lib.QTX_F32 if dtype == np.float32 else _lib.QTX_F64, Od.data_ptr(),
              md.data_ptr(), rd.data_ptr() if weights else None, ns, np_, 0, S.data_ptr(), None, 0)
    S = S.cpu().numpy()
    assert np.array_equal(S, S.T)
    assert np.all(np.abs(S - A.T @ A) <= (ns + 8) * 2.0**-53 * (np.abs(A).T @ np.abs(A)))


@pytest.mark.parametrize("np_", [511, 512, 513])
def test_solve_on_both_sides_of_the_line(np_):
    """The shifted SR solve with S from either route: 16 (ns + np) u cond."""
    rng = np.random.default_rng(np_)
    ns = 700
    O, e = rng.standard_normal((ns, np_)), rng.standard_normal(ns)
    mean = O.mean(0)
    A = (O - mean) / np.sqrt(ns)
    x = qtx.optimizer.solve_step(*(torch.as_tensor(v, device="cuda") for v in (O, mean, e)),
                                 qtx.optimizer.lstsq_shift_eig(rshift=1e-6, ashift=0.0)).cpu().numpy()
    ref = osr.lstsq_shift_eig(A, e, rshift=1e-6, ashift=0.0)
    lam = np.linalg.eigvalsh(A.T @ A) + 1e-6 * np.trace(A.T @ A)
    assert np.linalg.norm(x - ref) <= 16 * (ns + np_) * 2.0**-53 * lam[-1] / lam[0] * np.linalg.norm(ref)
