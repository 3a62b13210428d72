"""The blocked Cholesky factorisation and its fused substitutions at the edges
of their tiles: 16-column groups, 64-column panels, 1024-column diagonal blocks.

The shifted solve is compared with the same solve in float64 on the CPU.
Tolerance: 8 (n + np) u cond(T + shift), u = 2^-53: the usual bounds of the
Gram sum (np terms) and of a Cholesky solve, with the condition number computed."""

import numpy as np
import pytest
import torch

import quantax_amd as qtx
from oracle import sr as osr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 48, 63, 64, 65, 128, 130, 272, 1000, 1023, 1024, 1025, 1090, 2113])
def test_shifted_solve(n):
    rng = np.random.default_rng(n)
    np_ = n + 1 + n // 8
    O = rng.standard_normal((n, np_)) * np.logspace(0, -1.5, n)[:, None]
    y = rng.standard_normal(n)
    Od = torch.as_tensor(O, device="cuda")
    mean = torch.zeros(np_, dtype=torch.float64, device="cuda")
    x = qtx.optimizer.solve_step(Od, mean, torch.as_tensor(y, device="cuda"),
                                 qtx.optimizer.minnorm_shift_eig(rshift=1e-6, ashift=1e-8, gram="fp64")).cpu().numpy()
    A = O / np.sqrt(n)
    ref = osr.minnorm_shift_eig(A, y, rshift=1e-6, ashift=1e-8)
    lam = np.linalg.eigvalsh(A @ A.T)
    shift = 1e-6 * lam.sum() + 1e-8
    cond = (lam[-1] + shift) / (max(lam[0], 0.0) + shift)
    err = np.linalg.norm(x - ref) / np.linalg.norm(ref)
    tol = 8 * (n + np_) * 2.0**-53 * cond
    print(f"n {n}: cond {cond:.1e} err {err:.2e} tol {tol:.2e}")
    assert err <= tol, (err, tol)
