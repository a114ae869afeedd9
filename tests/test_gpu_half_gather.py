"""The paired gather of half-storage cells: rays along the last cells of each z row (whose ceil wraps),
exact integer coordinates, and grids one and two cells high, against the float32 kernel on the same
(exactly representable) values -- the same bits."""
import pytest
import torch

from plenoxels_amd import pack_occupancy
from plenoxels_amd.render import render_rays
from util import say

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("Z", [1, 2, 3, 8, 33])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("occupied", [False, True])  # one ray per wave; with 2^14 rays or more, two
def test_half_gather_equals_float32(Z, dtype, occupied):
    say("half gather", Z, dtype, occupied)
    g = torch.Generator().manual_seed(Z)
    dims, pd, R, S = (5, 6, Z), 0.5, (1 << 14) + 1 if occupied else 257, 70
    grid = (torch.rand(*dims, 4, generator=g) * 1.2 - 0.1).to(dtype)
    size = torch.tensor(dims) * pd
    a, b = (torch.rand(R, 3, generator=g) * size * 1.2 - 0.1 * size for _ in range(2))
    a[::3, 2] = b[::3, 2] = (Z - 1) * pd + 0.4 * pd  # in the wrapping slab
    a[1::3] = (a[1::3] / pd).round() * pd             # integer coordinates, a cell per sample along x
    d = torch.nn.functional.normalize(b - a, dim=1)
    d[1::3] = torch.tensor([1.0, 0.0, 0.0])
    o = a - d * 0.5 * S * 0.1
    o[1::3] = a[1::3] - d[1::3] * 2.0
    bits = pack_occupancy(torch.ones(dims, dtype=torch.bool, device=DEV)) if occupied else None
    kw = dict(num_samples=S, delta_step=0.125, grid_min=(0.0, 0.0, 0.0), points_distance=pd, interp="trilinear",
              occupancy=bits)
    half = render_rays(grid.to(DEV), o.to(DEV), d.to(DEV), **kw)
    full = render_rays(grid.float().to(DEV), o.to(DEV), d.to(DEV), **kw)
    assert full.abs().max() > 0 and torch.equal(half, full)
