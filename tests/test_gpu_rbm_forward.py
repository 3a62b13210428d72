"""The RBM forward at the edges of its loops: hidden units around multiples of 64 (a
lane's registers come in powers of two, the last ones partly or wholly empty), sites
around the batches of 1, 2, 4 and 8 rows.

Against float64 numpy.  Tolerance: a unit's sum of N + 1 terms in the model's type is
off by (N + 2) u sum |terms|, log cosh (slope at most 1) by a few u of its value, the
sum over the units by M / 64 + 6 roundings."""
import numpy as np
import pytest
import torch

import quantax_amd as qtx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 63, 64, 65, 127, 128, 129, 191, 193, 257, 400, 512, 513, 1000, 1024])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_forward(M, dtype):
    for N in (2, 7, 8, 9, 15, 17, 33):
        qtx.sites.Chain(N)
        model = qtx.model.RBM_Dense(M, dtype=dtype, init_std=0.2, seed=N)
        rng = np.random.default_rng(M + N)
        s = rng.choice([-1, 1], (37, N)).astype(np.int8)
        got, h = model.logpsi(torch.as_tensor(s, device="cuda"), h_out=True)
        th = model.theta.cpu().numpy().astype(np.float64)
        W, b = th[: M * N].reshape(M, N), th[M * N:]
        ref = s @ W.T + b
        u = 2.0**-24 if dtype == np.float32 else 2.0**-53
        dh = (N + 2) * u * (np.abs(W).sum(1) + np.abs(b))
        assert np.all(np.abs(h.cpu().numpy() - ref) <= dh), N
        lc = np.abs(ref) + np.log1p(np.exp(-2 * np.abs(ref))) - np.log(2.0)
        tol = dh.sum() + (8 + M // 64 + 6) * u * (np.abs(ref) + 1).sum(1)
        assert np.all(np.abs(got.cpu().numpy() - lc.sum(1)) <= tol), N
