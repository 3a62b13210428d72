"""Which way a few configurations of a projected RBM go: the kernels without images, or
images -> forward -> projection where one workgroup would take a large group's tiles in
turn."""
from types import SimpleNamespace

import numpy as np
import pytest
import torch

import quantax_amd as qtx

from .test_symm_route import _symm


# the sides measured as at least a tenth apart, 1 to 64 configurations
@pytest.mark.parametrize("L,M,z2,nperm,ns,images", [
    (8, 64, 1, 512, 1, True), (8, 64, 1, 512, 16, True), (8, 64, 1, 512, 32, False), (8, 36, 1, 512, 4, True),
    (8, 36, 1, 512, 30, False), (8, 8, 1, 512, 16, False), (8, 64, 0, 512, 16, True), (8, 36, 0, 512, 8, True),
    (8, 50, 0, 512, 64, False), (8, 4, 0, 512, 1, False), (7, 64, 0, 392, 16, True), (7, 36, 0, 392, 1, True),
    (7, 64, 0, 392, 64, False), (6, 50, 0, 288, 1, False), (6, 64, 1, 288, 32, False), (8, 64, 1, 64, 1, False),
    (4, 64, 1, 128, 1, False), (8, 64, 0, 512, 1000, False)])
def test_the_faster_side(L, M, z2, nperm, ns, images):
    assert _symm(L, nperm, z2).images_faster(SimpleNamespace(M=M), ns) == images


@pytest.mark.gpu
@pytest.mark.parametrize("z2", [0, 1, -1])
def test_both_sides_agree(z2):
    """As tests/test_gpu_symm_fused.py: float64 sums of 64 units and 512 or 1024 images."""
    symm = _symm(8, 512, z2)
    model = qtx.model.RBM_Dense(64, dtype=np.float64, init_std=0.05, seed=1)
    state = qtx.state.Variational(model, symm=symm)
    g = torch.Generator(device="cuda").manual_seed(5)
    s = torch.where(torch.rand((4, 64), generator=g, device="cuda").argsort(1) < 32, 1, -1).to(torch.int8)
    assert symm.images_faster(model, 4)
    psi, (sg, la) = state(s), symm.rbm_logpsi(model, s)
    big = model.logpsi(symm.images(s)).view(4, -1).max(1).values
    ok = la - big > np.log(1e-8)  # not cancelled to round-off
    assert torch.equal(psi.sign[ok], sg[ok])
    assert bool(((psi.logabs - la).abs() <= 1e-12 * la.abs().clamp(min=1) + 1e-13 * torch.exp(big - la))[ok].all())
