"""Column sums of narrow matrices, whose rows share a wave: the numbers of lanes per
row (columns up to 4, 8, ..., 128, then 256 a workgroup), the masked rows at a chunk's
end and the parts of 2048 weights.

Against float64 numpy.  Tolerance: a sum of n terms in any order is off by at most
n u sum |terms|, u = 2^-53, and each term carries a few roundings more."""
import numpy as np
import pytest
import torch

import quantax_amd as qtx
from quantax_amd import _lib

pytestmark = pytest.mark.gpu
EDGES = [1, 3, 4, 5, 8, 9, 16, 17, 31, 32, 33, 64, 65, 127, 128, 129, 257]


@pytest.mark.parametrize("np_", EDGES)
@pytest.mark.parametrize("ns", [1, 7, 130, 1025, 33000])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_means(ns, np_, dtype):
    rng = np.random.default_rng(ns + np_)
    O = (rng.standard_normal((ns, np_)) + 0.5).astype(dtype)
    flat = torch.zeros(ns * np_ + 1, dtype=torch.float32 if dtype == np.float32 else torch.float64, device="cuda")
    flat[1:] = torch.as_tensor(O, device="cuda").reshape(-1)  # rows at any element's alignment
    mean = torch.empty(np_, dtype=torch.float64, device="cuda")
    _lib.call("qtx_colmean", _lib.stream(), _lib.QTX_F32 if dtype == np.float32 else _lib.QTX_F64,
              flat[1:].data_ptr(), ns, np_, mean.data_ptr())
    X = O.astype(np.float64)
    assert np.all(np.abs(mean.cpu().numpy() - X.mean(0)) <= 2 * (ns + 4) * 2.0**-53 * np.abs(X).sum(0) / ns)


@pytest.mark.parametrize("ns,np_", [(300, 1), (300, 4), (2100, 5), (4099, 16), (700, 33), (3000, 65), (600, 129),
                                    (270000, 3)])
@pytest.mark.parametrize("weights", [False, True])
def test_weighted_sums(ns, np_, weights):
    """x = (S + shift)^-1 F with F = Obar^T e and a shift of ten traces: x = F / shift up
    to a tenth, so an error of F comes through and the solve adds a few u."""
    rng = np.random.default_rng(ns + np_)
    O = rng.standard_normal((ns, np_))
    r = rng.random(ns) + 0.5
    e = rng.standard_normal(ns)
    mean = O.mean(0)
    A = (O - mean) * np.sqrt((r if weights else np.ones(ns)) / ns)[:, None]
    S = A.T @ A
    ref = np.linalg.solve(S + 10.0 * np.trace(S) * np.eye(np_), A.T @ e)
    x = qtx.optimizer.solve_step(torch.as_tensor(O, device="cuda"), torch.as_tensor(mean, device="cuda"),
                                 torch.as_tensor(e, device="cuda"),
                                 qtx.optimizer.lstsq_shift_eig(rshift=10.0, ashift=0.0),
                                 torch.as_tensor(r, device="cuda") if weights else None).cpu().numpy()
    tol = 4 * (ns + np_ + 8) * 2.0**-53 * (np.abs(A).T @ np.abs(e)).max() / (10.0 * np.trace(S))
    assert np.abs(x - ref).max() <= tol
