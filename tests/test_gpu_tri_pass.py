"""The one-read triangle passes of the solver: the symmetric product of the
Lanczos steps (n >= 4608) and P^T (P x) of the Chebyshev terms (n >= 2560), on
both sides of their lines, at the edges of their column classes (n <= 4096,
n <= 8192, above) and at odd n (rows that end inside a pair of columns and are
not 16-byte aligned), with the register forms of the Lanczos step.

O = sqrt(n) H1 D H2 with reflections H1, H2 and a diagonal D of known singular
values, so the answer has a closed form in float64 at any n."""

import numpy as np
import pytest
import torch

import quantax_amd as qtx
from oracle import sr as osr

pytestmark = pytest.mark.gpu


def _reflector(gen, n):
    v = torch.randn(n, dtype=torch.float64, device="cuda", generator=gen)
    return v / v.norm()


@pytest.mark.parametrize("n", [2559, 2560, 2561, 3073, 4096, 4099, 4607, 4608, 8192, 8193, 9001])
def test_solve_closed_form(n):
    gen = torch.Generator(device="cuda").manual_seed(n)
    np_ = n + 7
    u, v = _reflector(gen, n), _reflector(gen, np_)
    lam = torch.logspace(0, -9, n, dtype=torch.float64, device="cuda")
    lam = lam[torch.randperm(n, device="cuda", generator=gen)]
    s = lam.sqrt()
    # H1 D H2 = D - 2 u (u.D) - 2 (D v) v + 4 (u.D.v) u v, D = [diag(s), 0]
    dv = s * v[:n]
    ud = torch.zeros(np_, dtype=torch.float64, device="cuda")
    ud[:n] = u * s
    O = torch.zeros(n, np_, dtype=torch.float64, device="cuda")
    O[torch.arange(n), torch.arange(n)] = s
    O -= 2 * torch.outer(u, ud) + 2 * torch.outer(dv, v) - 4 * (u @ dv) * torch.outer(u, v)
    O *= n**0.5
    y = torch.randn(n, dtype=torch.float64, device="cuda", generator=gen)
    mean = torch.zeros(np_, dtype=torch.float64, device="cuda")
    rtol = 1e-4
    x = qtx.optimizer.solve_step(O, mean, y, qtx.optimizer.auto_pinv_eig(rtol=rtol, gram="fp64"))
    info = qtx.optimizer.last_solve_info()
    assert info["path"] == "chebyshev", info
    inv = torch.as_tensor(osr.eigs_inv(lam.cpu().numpy(), rtol=rtol)).cuda()
    z = torch.zeros(np_, dtype=torch.float64, device="cuda")
    z[:n] = s * inv * (y - 2 * u * (u @ y))
    ref = z - 2 * v * (v @ z)
    err = ((x - ref).norm() / ref.norm()).item()
    print(f"n {n}: err {err:.2e}")
    assert err < 1e-9, err  # the bound of the other Chebyshev tests
