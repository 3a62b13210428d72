"""Column means and the weighted column sums x = Obar^T y (the last product of
a MinSR solve) at the edges of their split: columns in fours and 256s, rows in
groups of 32 per wave pass, 16 per chunk and 512 weights per part.

Against float64 numpy.  Tolerance: a sum of n terms in any order is off by at
most n u sum |terms|, u = 2^-53, and each term carries a few roundings more."""

import numpy as np
import pytest
import torch

import quantax_amd as qtx
from quantax_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns,np_", [(1, 1), (1, 5), (3, 255), (15, 256), (17, 257), (31, 1022), (33, 4), (512, 3),
                                    (513, 260), (1024, 272), (5000, 2), (40000, 3), (300, 3001)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_column_sums(ns, np_, dtype):
    rng = np.random.default_rng(ns * 7 + np_)
    O = (rng.standard_normal((ns, np_)) + 0.5).astype(dtype)
    Od = torch.as_tensor(O, device="cuda")
    mean = torch.empty(np_, dtype=torch.float64, device="cuda")
    code = _lib.QTX_F32 if dtype == np.float32 else _lib.QTX_F64
    _lib.call("qtx_colmean", _lib.stream(), code, Od.data_ptr(), ns, np_, mean.data_ptr())
    X = O.astype(np.float64)
    u = 2.0**-53
    assert np.all(np.abs(mean.cpu().numpy() - X.mean(0)) <= 2 * (ns + 4) * u * np.abs(X).sum(0) / ns)


@pytest.mark.parametrize("ns,np_", [(2, 2), (3, 255), (15, 256), (17, 259), (31, 1022), (513, 516), (700, 703)])
@pytest.mark.parametrize("weights", [False, True])
def test_weighted_sums(ns, np_, weights):
    """x = Obar^T z, with z from the same solve in float64 (a well-conditioned
    shift, so that z is known to a few ulps of its norm)."""
    rng = np.random.default_rng(ns + np_)
    O = rng.standard_normal((ns, np_))
    r = rng.random(ns) + 0.5 if weights else None
    e = rng.standard_normal(ns)
    mean = O.mean(0)
    A = (O - mean) * np.sqrt((r if weights else np.ones(ns)) / ns)[:, None]
    shift = 10.0 * np.trace(A @ A.T)
    z = np.linalg.solve(A @ A.T + shift * np.eye(ns), e)
    ref = A.T @ z
    x = qtx.optimizer.solve_step(torch.as_tensor(O, device="cuda"), torch.as_tensor(mean, device="cuda"),
                                 torch.as_tensor(e, device="cuda"),
                                 qtx.optimizer.minnorm_shift_eig(rshift=10.0, ashift=0.0),
                                 None if r is None else torch.as_tensor(r, device="cuda")).cpu().numpy()
    tol = 16 * (ns + np_) * 2.0**-53 * (np.abs(A).T @ np.abs(z)).max()
    assert np.abs(x - ref).max() <= tol
