"""Which way a batch of a projected RBM goes: the kernels without images, or images ->
forward -> projection for small groups in large batches."""
from types import SimpleNamespace

import numpy as np
import pytest
import torch

import quantax_amd as qtx


def _symm(L, nperm, z2):
    N = L * L
    qtx.sites.Square(L, Nparticles=(N // 2, N - N // 2))
    rng = np.random.default_rng(nperm)
    perm = np.stack([np.arange(N)] + [rng.permutation(N) for _ in range(nperm - 1)])
    return qtx.symmetry.Symmetry(Z2_inversion=z2, perm=perm, character=np.ones(nperm))


# the sides measured as at least a tenth apart, 4096 to 131072 configurations
@pytest.mark.parametrize("L,M,z2,nperm,ns,images", [
    (4, 16, 1, 1, 16384, True), (4, 16, 0, 2, 131072, True), (4, 16, 1, 2, 16384, False), (6, 12, 0, 3, 16384, False),
    (6, 36, 1, 1, 8192, True), (6, 36, 1, 1, 4096, False), (6, 36, 0, 2, 16384, True), (6, 36, 1, 2, 131072, False),
    (6, 36, 0, 4, 131072, False), (6, 64, 1, 1, 8192, True), (6, 64, 0, 3, 131072, True), (6, 64, 1, 2, 131072, True),
    (6, 64, 1, 3, 131072, False), (8, 20, 0, 2, 131072, False), (8, 64, 1, 1, 4096, True), (8, 64, 1, 1, 2048, False),
    (8, 64, 0, 2, 8192, True), (8, 64, 0, 4, 131072, False), (8, 64, 1, 8, 131072, False)])
def test_the_faster_side(L, M, z2, nperm, ns, images):
    assert _symm(L, nperm, z2).images_faster(SimpleNamespace(M=M), ns) == images


@pytest.mark.parametrize("L,M", [(2, 1), (3, 64), (8, 1), (8, 64)])
def test_large_groups_and_small_batches_stay(L, M):
    assert not _symm(L, 16, 0).images_faster(SimpleNamespace(M=M), 10**6)
    assert not _symm(L, 8, 1).images_faster(SimpleNamespace(M=M), 10**6)
    assert not _symm(L, 1, 1).images_faster(SimpleNamespace(M=M), 1024)


@pytest.mark.gpu
@pytest.mark.parametrize("z2,nperm", [(1, 1), (-1, 1), (0, 2)])
def test_both_sides_agree(z2, nperm):
    """As tests/test_gpu_symm_fused.py: float64 sums of 36 units and two images."""
    symm = _symm(6, nperm, z2)
    model = qtx.model.RBM_Dense(36, dtype=np.float64, init_std=0.05, seed=1)
    state = qtx.state.Variational(model, symm=symm)
    g = torch.Generator(device="cuda").manual_seed(5)
    s = torch.where(torch.rand((8192, 36), generator=g, device="cuda").argsort(1) < 18, 1, -1).to(torch.int8)
    assert symm.images_faster(model, 8192)
    psi, (sg, la) = state(s), symm.rbm_logpsi(model, s)
    big = model.logpsi(symm.images(s)).view(8192, -1).max(1).values
    ok = la - big > np.log(1e-8)  # not cancelled to round-off
    assert torch.equal(psi.sign[ok], sg[ok])
    assert bool(((psi.logabs - la).abs() <= 1e-12 * la.abs().clamp(min=1) + 1e-13 * torch.exp(big - la))[ok].all())
