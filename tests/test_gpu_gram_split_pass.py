"""The pass that splits Obar into bf16 parts, eight columns per thread: np around
multiples of eight, 64 and 2048, rows past n, both input types, with and
without weights; bit for bit hi = bf16(x), lo = bf16(x - hi) of the
single-precision x, in the layout of 32 hi and their 32 lo per row."""

import pytest
import torch

from quantax_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,np_", [(1, 2), (5, 7), (5, 8), (7, 9), (3, 63), (3, 64), (3, 65), (130, 2047), (9, 2048),
                                   (9, 2057), (128, 4100)])
@pytest.mark.parametrize("dtype,weights", [(torch.float32, True), (torch.float64, False)])
def test_split(n, np_, dtype, weights):
    gen = torch.Generator(device="cuda").manual_seed(n * np_)
    O = torch.randn(n, np_, device="cuda", generator=gen, dtype=dtype)
    mean = O.mean(0, dtype=torch.float64) * 0.5
    r = torch.rand(n, device="cuda", dtype=torch.float64, generator=gen) + 0.5
    nws = int(_lib.lib().qtx_gram_ws_bytes(n, np_, 2))
    ws = torch.full((nws,), 0x55, dtype=torch.uint8, device="cuda")
    T = torch.empty(n, n, dtype=torch.float64, device="cuda")
    _lib.call("qtx_gram", _lib.stream(), _lib.QTX_F32 if dtype == torch.float32 else _lib.QTX_F64, O.data_ptr(),
              mean.data_ptr(), r.data_ptr() if weights else None, n, np_, 2, T.data_ptr(), ws.data_ptr(), nws)
    rows, kpad = (n + 127) // 128 * 128, (np_ + 63) // 64 * 64
    parts = ws.view(torch.bfloat16)[: 2 * rows * kpad].view(rows, kpad // 32, 2, 32)
    x = torch.zeros(rows, kpad, dtype=torch.float32, device="cuda")
    w = r if weights else torch.ones_like(r)
    x[:n, :np_] = ((O.double() - mean) * torch.sqrt(w * (1.0 / n))[:, None]).float()
    hi = x.bfloat16()
    lo = (x - hi.float()).bfloat16()
    assert torch.equal(parts[:, :, 0].reshape(rows, kpad), hi)
    assert torch.equal(parts[:, :, 1].reshape(rows, kpad), lo)
