"""The two-rays-per-wavefront forward (occupancy given, up to 512 samples per ray, at least 2^14 rays) against the
one-ray kernel: the same bits, outputs and saved state, for every chunk count, odd batches, rays
with at most and with more than 32 kept samples, and early termination.  Without occupancy the
one-ray kernel runs, so an occupancy of ones compares the two."""
import ctypes

import pytest
import torch

from plenoxels_amd import MarchConfig, _lib, pack_occupancy
from plenoxels_amd.render import _grid_struct, _rays_struct
from test_gpu_bins import _scene
from util import say

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _forward(grid, o, d, cfg, bits):
    L = _lib.lib()
    R, n = o.shape[0], int(L.pxl_aux_floats(cfg.num_samples))
    out, aux = torch.empty(R, 4, device=DEV), torch.zeros(R, n, device=DEV)
    g, m, r = _grid_struct(grid, bits), cfg.to_struct(), _rays_struct(o, d)
    for a in (aux, None):
        _lib.check(L.pxl_render_fwd(ctypes.byref(g), ctypes.byref(m), ctypes.byref(r), _lib.ptr(out), _lib.ptr(a),
                                    _lib.stream_handle(DEV)))
        if a is not None:
            first = out.clone()
    assert torch.equal(first, out)
    # only the groups that were walked are defined
    ng = aux[:, 1].contiguous().view(torch.int32)
    used = torch.arange(n, device=DEV)[None, :] < 2 + 2 * ng[:, None]
    return out, torch.where(used, aux, torch.zeros_like(aux)).view(torch.int32)


@pytest.mark.parametrize("S", [1, 64, 65, 128, 129, 256, 257, 512])
@pytest.mark.parametrize("interp,t_stop,dtype", [("nearest", 0.0, torch.float32), ("trilinear", 0.05, torch.float32),
                                                 ("trilinear", 0.0, torch.float16), ("nearest", 0.05, torch.bfloat16)])
@pytest.mark.parametrize("dims", [(20, 20, 20), (70, 33, 40)])  # ~17 and ~40 samples per ray inside
def test_pair_forward_equals_one_ray_forward(S, interp, t_stop, dtype, dims):
    say("pair forward", S, interp, t_stop, dtype, dims)
    R = (1 << 14) + 7
    grid, o, d, gmin, pd, delta, _ = _scene(dims, R, S, 7)
    grid = grid.to(dtype).to(DEV)
    o[-1], d[-1] = o[0] + 100.0, d[0]  # a ray that misses
    ones = pack_occupancy(torch.ones(dims, dtype=torch.bool, device=DEV))
    cfg = MarchConfig(S, delta, gmin, pd, interp, 0.0, t_stop)
    for n in (R, R - 1, 1 << 14, (1 << 14) + 1):  # 2^14 is the smallest batch taken in pairs
        a, ax = _forward(grid, o[:n].contiguous().to(DEV), d[:n].contiguous().to(DEV), cfg, None)
        b, bx = _forward(grid, o[:n].contiguous().to(DEV), d[:n].contiguous().to(DEV), cfg, ones)
        assert torch.equal(a, b) and torch.equal(ax, bx)


@pytest.mark.parametrize("S", [300, 512])
@pytest.mark.parametrize("interp,t_stop", [("nearest", 0.3), ("trilinear", 0.3), ("trilinear", 0.0)])
def test_pair_forward_of_long_rays(S, interp, t_stop):
    """Rays that keep a hundred and more samples: both of a pair, one, or neither stopped by their first
    group (alpha differs by regions), so that classification ends early for some pairs and goes on for
    the rays of others; the last ray alone in its pair keeps more than 32 samples."""
    say("pair forward, long rays", S, interp, t_stop)
    R, dims = (1 << 14) + 1, (150, 161, 140)
    grid, o, d, gmin, pd, delta, _ = _scene(dims, R, S, 8)
    grid[:80, ..., 3] *= 0.02
    grid = grid.to(DEV)
    d[-1] = torch.tensor([1.0, 0.0, 0.0])  # along x through the middle: ~125 samples, the thin ones first
    o[-1] = torch.tensor(gmin) + torch.tensor(dims) * (pd / 2) - d[-1] * (delta * S / 2)
    o, d = o.to(DEV), d.to(DEV)
    ones = pack_occupancy(torch.ones(dims, dtype=torch.bool, device=DEV))
    cfg = MarchConfig(S, delta, gmin, pd, interp, 0.0, t_stop)
    a, ax = _forward(grid, o, d, cfg, None)
    b, bx = _forward(grid, o, d, cfg, ones)
    assert torch.equal(a, b) and torch.equal(ax, bx)
    groups, stopped = ax[:, 1], ax[:, 0] < S
    assert (groups > 1).any() and groups[-1] > 1
    assert t_stop == 0.0 or (stopped[0:-1:2] & stopped[1::2]).any() and (stopped[0:-1:2] ^ stopped[1::2]).any()
