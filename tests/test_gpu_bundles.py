"""The nearest train step's cell sums of neighbouring rays (no occupancy, up to 256 samples) against
the plain chain's autograd: whole views whose workgroups' rays share cells, odd batches, more cells
than the table holds, and batches where only some workgroups are bundles."""
import pytest
import torch

from oracle import plain
from plenoxels_amd import MarchConfig, pack_occupancy, train_step
from util import grad_close, say

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("S", [1, 64, 128, 200, 256])
@pytest.mark.parametrize("R,step,kind", [(1, 0.3, "fan"), (7, 0.3, "fan"), (8, 0.05, "fan"), (403, 0.3, "fan"),
                                         (403, 0.3, "mixed"), (403, 0.0, "same")])
def test_bundle_gradient(S, R, step, kind):
    """step: cells between neighbouring rays.  delta of half a cell down the long axis: runs, and with
    S = 256 eight rays reach more cells than the table has slots."""
    say("bundles", S, R, step, kind)
    dims, pd = (150, 60, 60), 0.1
    g = torch.Generator().manual_seed(S + R)
    grid = torch.rand(*dims, 4, generator=g) * 1.2 - 0.1
    grid[..., 3] *= 0.05
    o = torch.tensor([[-0.5, 2.0, 2.0]]) + torch.arange(R).unsqueeze(1) * torch.tensor([[0.0, step * pd / 4, step * pd]]) % 2.0
    d = torch.nn.functional.normalize(torch.tensor([[1.0, 0.03, 0.11]]), dim=1).expand(R, 3).contiguous()
    if kind == "mixed":  # every other group of eight far apart
        far = (torch.arange(R) // 8) % 2 == 1
        o = torch.where(far.unsqueeze(1), o + torch.rand(R, 3, generator=g) * 3, o)
    # identical rays get one target: with random ones their 403 terms of a cell cancel to 1% and less of
    # the terms' size, and float32's 1e-6 of a term is then above 1e-4 of the sum
    tgt = torch.rand(1 if kind == "same" else R, 4, generator=g).expand(R, 4).contiguous()
    cfg = MarchConfig(S, pd * 0.7, (0.0, 0.0, 0.0), pd, "nearest")
    grad = torch.zeros(*dims, 4, device=DEV)
    train_step(grid.to(DEV), grad, cfg=cfg, origins=o.contiguous().to(DEV), dirs=d.to(DEV), targets=tgt.to(DEV))
    ref = grid.double().requires_grad_(True)
    out = plain.render(ref, o, d, num_samples=S, delta_step=pd * 0.7, gmin=torch.zeros(3), points_distance=pd,
                       interp="nearest", div_mode="reciprocal")
    ((out - tgt.double()) ** 2).mean().backward()
    ok, info = grad_close(grad.cpu(), ref.grad)
    say("  ", info)
    assert ok, info


@pytest.mark.parametrize("S", [40, 128, 256])
@pytest.mark.parametrize("dtype,empty,t_stop", [(torch.float32, 0.95, 0.0), (torch.bfloat16, 0.5, 0.1),
                                                (torch.float16, 1.0, 0.0)])
def test_bundle_gradient_in_empty_space(S, dtype, empty, t_stop):
    """Samples whose cell takes no gradient (alpha below zero) take no slot of the table; rays that stop
    early leave some waves with few samples; a grid that is all empty leaves nothing to add."""
    say("bundles in empty space", S, dtype, empty, t_stop)
    dims, pd, R = (70, 60, 50), 0.1, 331
    g = torch.Generator().manual_seed(S)
    grid = torch.rand(*dims, 4, generator=g) * 1.2 - 0.1
    grid[..., 3] = torch.where(torch.rand(dims, generator=g) < empty, -0.1, grid[..., 3].abs() * 0.5)
    grid = grid.to(dtype).float()
    o = torch.tensor([[-0.5, 2.0, 2.0]]) + torch.arange(R).unsqueeze(1) * torch.tensor([[0.0, 0.01, 0.03]]) % 2.0
    d = torch.nn.functional.normalize(torch.tensor([[1.0, 0.03, 0.11]]), dim=1).expand(R, 3).contiguous()
    tgt = torch.rand(R, 4, generator=g)
    cfg = MarchConfig(S, pd * 0.4, (0.0, 0.0, 0.0), pd, "nearest", 0.0, t_stop)
    grad = torch.zeros(*dims, 4, device=DEV)
    train_step(grid.to(dtype).to(DEV), grad, cfg=cfg, origins=o.contiguous().to(DEV), dirs=d.to(DEV), targets=tgt.to(DEV))
    if empty == 1.0:
        assert grad.abs().max() == 0
        return
    # with an occupancy of ones the samples go straight to the gradient: the same terms in another order
    want = torch.zeros(*dims, 4, device=DEV)
    ones = pack_occupancy(torch.ones(dims, dtype=torch.bool, device=DEV))
    train_step(grid.to(dtype).to(DEV), want, cfg=cfg, origins=o.contiguous().to(DEV), dirs=d.to(DEV), targets=tgt.to(DEV),
               occupancy=ones)
    ok, info = grad_close(grad.cpu(), want.cpu())
    say("  ", info)
    assert ok and want.abs().max() > 0, info
