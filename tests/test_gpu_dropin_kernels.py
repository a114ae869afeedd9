"""The drop-ins' column minimum, nearest gather and scatter, and TV gradient at the sizes and values
where their vector paths can go wrong."""
import pytest
import torch

from oracle import plain
from plenoxels_amd.grid_functions import get_nearest_voxels
from plenoxels_amd.optim import tv_loss
from plenoxels_amd.ray_sampling import normalize_samples_for_indecies
from util import grad_close, say

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("n,offset", [(1, 0), (2, 0), (3, 0), (5, 0), (341, 0), (1025, 0), (4099, 0), (2000003, 0),
                                      (341, 1), (4099, 2), (100001, 3)])
@pytest.mark.parametrize("shift", [-3.0, 0.0, 5.0])  # minima negative, of mixed sign, positive
def test_column_minimum(n, offset, shift):
    """offset floats into a buffer: the array is then 4-byte aligned only."""
    say("column minimum", n, offset, shift)
    g = torch.Generator().manual_seed(n)
    buf = (torch.randn(3 * n + offset, generator=g) + shift).to(DEV)
    coords = buf[offset:].reshape(n, 3)
    p = torch.zeros(1, 3, device=DEV)
    got = normalize_samples_for_indecies(coords, p, 1.0)
    assert torch.equal(got[0], -coords.min(0)[0])


@pytest.mark.parametrize("N", [1, 63, 64, 65, 255, 257, 10007])
@pytest.mark.parametrize("spacing", [0.05, 1.7])  # runs of one cell, and none
def test_nearest_gather_and_scatter(N, spacing):
    say("nearest gather/scatter", N, spacing)
    dims = (7, 30, 11)
    g = torch.Generator().manual_seed(N)
    grid = torch.rand(*dims, 4, generator=g)
    n = torch.rand(N, 3, generator=g) * 0.01 + (torch.arange(N).unsqueeze(1) * spacing) % 40 - 5  # in and out of the grid
    if N > 60:  # beyond 32-bit indices, and exact halves
        n[3] = torch.tensor([3.0e9, -3.0e9, 2.5])
        n[4] = torch.tensor([-0.5, 0.5, 1.5])
        n[5] = torch.tensor([1.0e9, -2.0e9, 7.0e18])
    up = torch.rand(N, 4, generator=g) - 0.5
    up[::5] = 0
    up[1::7, :3] = 0
    leaf = grid.to(DEV).requires_grad_(True)
    vals, mask = get_nearest_voxels(n.to(DEV), leaf)
    (vals * up.to(DEV)).sum().backward()
    idx = n.round().to(torch.long)
    want_mask = plain.find_out_of_bound(idx, dims)
    w = torch.stack([torch.remainder(idx[:, a], dims[a]) for a in range(3)], 1)
    assert torch.equal(mask.cpu(), want_mask)
    assert torch.equal(vals.detach().cpu(), grid[w[:, 0], w[:, 1], w[:, 2]])
    want = torch.zeros(*dims, 4, dtype=torch.float64)
    want.index_put_((w[:, 0], w[:, 1], w[:, 2]), up.double(), accumulate=True)
    # a cell sums up to a few hundred float32 terms of size <= 1/2: 2^-24 of their running sum each
    assert (leaf.grad.cpu().double() - want).abs().max().item() <= 1e-4


@pytest.mark.parametrize("dims", [(1, 1, 2), (2, 5, 65), (40, 9, 70)])
def test_tv_gradient_with_upstream(dims):
    say("tv gradient", dims)
    g = torch.Generator().manual_seed(sum(dims))
    base = torch.rand(*dims, 4, generator=g)
    leaf = base.to(DEV).requires_grad_(True)
    (tv_loss(leaf) * 0.37).backward()
    ref = base.double().requires_grad_(True)
    (plain.tv_loss(ref) * 0.37).backward()
    ok, info = grad_close(leaf.grad.cpu(), ref.grad, rel=1e-5)
    assert ok, info
    strided = base.to(DEV).transpose(0, 1).requires_grad_(True)  # not contiguous
    (tv_loss(strided) * 0.37).backward()
    ref = base.transpose(0, 1).double().requires_grad_(True)
    (plain.tv_loss(ref) * 0.37).backward()
    ok, info = grad_close(strided.grad.cpu(), ref.grad, rel=1e-5)
    assert ok, info
