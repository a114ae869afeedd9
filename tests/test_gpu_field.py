"""The occupancy + TV pass at the sizes where its walk can go wrong: rows and planes that do not fill
a tile, a slab, a wave or a workgroup, single cells, and more units than resident workgroups."""
import pytest
import torch

from oracle import plain
from plenoxels_amd import alpha_occupancy
from plenoxels_amd.optim import tv_sumsq
from util import say

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("dims", [(1, 1, 1), (1, 9, 64), (2, 3, 65), (8, 8, 8), (9, 4, 63), (17, 5, 128), (33, 12, 129),
                                  (64, 7, 5), (130, 70, 200), (72, 260, 260)])
@pytest.mark.parametrize("interp", ["nearest", "trilinear"])
def test_field_pass(dims, interp):
    say("field pass", dims, interp)
    g = torch.Generator(device=DEV).manual_seed(sum(dims))
    grid = torch.rand(*dims, 4, device=DEV, generator=g) - 0.6
    grid[0, 0, 0, 3] = -0.0
    occ = grid[..., 3] >= 0
    want = plain.occupancy_to_bits((plain.dilate_cells(occ) if interp == "trilinear" else occ).cpu())
    d = grid.double()
    # float32 differences and squares (one rounding each, 2^-24), summed in float64
    tv = sum(((d.narrow(a, 1, n - 1) - d.narrow(a, 0, n - 1)) ** 2).sum() for a, n in enumerate(dims)).item()
    s = torch.full((1,), 2.0, dtype=torch.float64, device=DEV)
    assert torch.equal(alpha_occupancy(grid, interp, s).cpu(), want)
    assert torch.equal(alpha_occupancy(grid, interp).cpu(), want)
    assert abs(s.item() - 2.0 - tv) <= 2.0 ** -22 * tv + 1e-14
    assert abs(tv_sumsq(grid).item() - tv) <= 2.0 ** -22 * tv
