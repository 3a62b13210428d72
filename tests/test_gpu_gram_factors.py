"""The Gram with reweighting factors and log-derivatives far from one: factors whose
products leave the range of float64, negative ones (no square root: NaN, so that the
update is refused), and O whose squares leave the range of float32.

Against float64 numpy: products of np terms, each operand rounded a few times."""
import numpy as np
import pytest
import torch

from quantax_amd import _lib

pytestmark = pytest.mark.gpu
GRAM = {"fp64": 0, "fp32": 1, "bf16x3": 2}


def gram(O, mean, r, mode):
    ns, np_ = O.shape
    Od, md = torch.as_tensor(O, device="cuda"), torch.as_tensor(mean, device="cuda")
    rd = None if r is None else torch.as_tensor(r, device="cuda")
    n = min(ns, np_)
    T = torch.full((n, n), float("nan"), dtype=torch.float64, device="cuda")
    wb = int(_lib.lib().qtx_gram_ws_bytes(ns, np_, GRAM[mode]))
    ws = torch.empty(max(wb, 1), dtype=torch.uint8, device="cuda")
    _lib.call("qtx_gram", _lib.stream(), _lib.QTX_F32 if O.dtype == np.float32 else _lib.QTX_F64, Od.data_ptr(),
              md.data_ptr(), _lib.ptr(rd), ns, np_, GRAM[mode], T.data_ptr(), ws.data_ptr(), wb)
    return T.cpu().numpy()


@pytest.mark.parametrize("ns", [40, 130])
def test_tiny_factors(ns):
    """r down to 1e-200: T_ij ~ sqrt(r_i r_j) to (np + 8) u, whatever r_i r_j is."""
    rng = np.random.default_rng(ns)
    O = rng.standard_normal((ns, 300))
    mean = O.mean(0)
    r = 10.0 ** rng.uniform(-200, 0, ns)
    r[:4] = 1e-200, 1e-190, 1e-180, 1.0
    f = np.sqrt(r / ns)
    A = O - mean
    T = gram(O, mean, r, "fp64") / f[:, None] / f[None, :]
    assert np.all(np.abs(T - A @ A.T) <= 308 * 2.0**-53 * (np.abs(A) @ np.abs(A).T))


@pytest.mark.parametrize("mode", ["fp64", "fp32", "bf16x3"])
@pytest.mark.parametrize("shape", [(20, 100), (100, 20)])
def test_negative_factors_are_nan(mode, shape):
    rng = np.random.default_rng(1)
    O = rng.standard_normal(shape)
    r = np.ones(shape[0])
    r[[3, 7]] = -1.0
    T = gram(O, O.mean(0), r, mode)
    if shape[0] < shape[1]:
        rows = np.isin(np.arange(20), [3, 7])
        assert np.isnan(T[rows]).all() and np.isnan(T[:, rows]).all()
        assert np.isfinite(T[np.ix_(~rows, ~rows)]).all()
    else:
        assert np.isnan(T).all()


@pytest.mark.parametrize("weights", [False, True])
def test_large_log_derivatives_in_fp32(weights):
    """|O| around 1e19: the squares are beyond float32, the squares over ns are not.
    Operands rounded to float32 and 256 products summed in it: (4 + 256) 2^-24."""
    rng = np.random.default_rng(2)
    ns, np_ = 200, 1000
    O = (1e19 * rng.uniform(-1, 1, (ns, np_))).astype(np.float32)
    mean = O.astype(np.float64).mean(0)
    r = rng.uniform(0.5, 1.0, ns) if weights else np.ones(ns)
    A = (O - mean) * np.sqrt(r / ns)[:, None]
    T = gram(O, mean, r if weights else None, "fp32")
    assert np.all(np.abs(T - A @ A.T) <= 260 * 2.0**-24 * (np.abs(A) @ np.abs(A).T))
