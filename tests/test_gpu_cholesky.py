"""The blocked Cholesky factorisation and its fused substitutions at the edges
of their tiles: 16-column groups, 64-column panels, the diagonal blocks (one up
to 6144 columns, 1024 and the rest beyond).

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


@pytest.mark.parametrize("n", [6143, 6144, 6145, 7300])
def test_shifted_solve_closed_form(n):
    """O = sqrt(n) H1 D H2 with reflections H1, H2 and known singular values, so
    x = H2 D^T (D^2 + shift)^-1 H1 y.  The same tolerance."""
    gen = torch.Generator(device="cuda").manual_seed(n)
    np_ = n + 7
    u, v = (torch.randn(k, dtype=torch.float64, device="cuda", generator=gen) for k in (n, np_))
    u, v = u / u.norm(), v / v.norm()
    s = torch.logspace(0, -2, n, dtype=torch.float64, device="cuda")
    s = s[torch.randperm(n, device="cuda", generator=gen)]
    dv, ud = s * v[:n], torch.zeros(np_, dtype=torch.float64, device="cuda")
    ud[:n] = u * s
    O = torch.zeros(n, np_, dtype=torch.float64, device="cuda")
    O[torch.arange(n), torch.arange(n)] = s
    O -= 2 * torch.outer(u, ud) + 2 * torch.outer(dv, v) - 4 * (u @ dv) * torch.outer(u, v)
    O *= n**0.5
    y = torch.randn(n, dtype=torch.float64, device="cuda", generator=gen)
    mean = torch.zeros(np_, dtype=torch.float64, device="cuda")
    x = qtx.optimizer.solve_step(O, mean, y, qtx.optimizer.minnorm_shift_eig(rshift=1e-8, ashift=1e-6, gram="fp64"))
    shift = 1e-8 * float((s * s).sum()) + 1e-6
    z = torch.zeros(np_, dtype=torch.float64, device="cuda")
    z[:n] = s / (s * s + shift) * (y - 2 * u * (u @ y))
    ref = z - 2 * v * (v @ z)
    err = float((x - ref).norm() / ref.norm())
    cond = (1.0 + shift) / (float((s * s).min()) + shift)
    tol = 8 * (n + np_) * 2.0**-53 * cond
    print(f"n {n}: cond {cond:.1e} err {err:.2e} tol {tol:.2e}")
    assert err <= tol
