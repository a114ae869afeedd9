"""GPU parity of the tile-binned trilinear scatter (pxl_train_step_work, pxl_render_bwd_work)
against the direct one (float atomics per corner) and the plain chain's autograd.

Both add the same products; only the order of the float32 sums differs, as for the corner blocks,
so the bars are theirs: 1e-5 relative between the two scatters, 1e-4 to autograd.
"""
import ctypes

import pytest
import torch

from oracle import plain
from plenoxels_amd import MarchConfig, _lib, occupancy_dilate, pack_occupancy, render, train_step
from plenoxels_amd.render import BIN_MIN_SAMPLES, _grid_struct, _rays_struct, render_rays
from util import grad_close, say

DEV = torch.device("cuda:0")
BASE = 2.0 ** -12


def _scene(dims, R, S, seed):
    """Rays through a grid of `dims` cells whose samples step about 1.2 cells and cross its faces."""
    g = torch.Generator().manual_seed(seed)
    pd = 0.1
    grid = torch.rand(*dims, 4, generator=g) * 1.2 - 0.1
    grid[..., 3] = grid[..., 3] * 0.2
    gmin = torch.tensor([-0.4, 0.3, 0.0])
    lo, size = gmin, torch.tensor(dims, dtype=torch.float32) * pd
    a = lo + (torch.rand(R, 3, generator=g) * 1.4 - 0.2) * size
    b = lo + torch.rand(R, 3, generator=g) * size
    d = torch.nn.functional.normalize(b - a, dim=1)
    delta = 0.12
    o = b - d * (delta * S / 2)
    return grid, o.contiguous(), d.contiguous(), tuple(gmin.tolist()), pd, delta, torch.rand(R, 4, generator=g)


def _train(grid, o, d, tgt, cfg, bits, work):
    L = _lib.lib()
    out, sq = torch.empty(o.shape[0], 4, device=DEV), torch.empty(o.shape[0], device=DEV)
    bsum = torch.empty(o.shape[0], device=DEV)
    # added to, not overwritten; every addition rounds to 2^-24 of the sum, so a small base costs
    # less than 1e-9 over the tens of additions a cell sees (a base of 0.25 would cost 1e-7 each)
    grad = torch.full(grid.shape, BASE, dtype=torch.float32, device=DEV)
    loss = _lib.Loss(targets=tgt.data_ptr(), grad_scale=0.5, beta_scale=1e-4, ray_sq_err=sq.data_ptr(),
                     ray_beta=bsum.data_ptr())
    g, m, r = _grid_struct(grid, bits), cfg.to_struct(), _rays_struct(o, d)
    _lib.check(L.pxl_train_step_work(ctypes.byref(g), ctypes.byref(m), ctypes.byref(r), ctypes.byref(loss),
                                     _lib.ptr(out), _lib.ptr(grad), _lib.ptr(work), 0 if work is None else work.numel(),
                                     _lib.stream_handle(DEV)))
    return out, sq, bsum, (grad - BASE).cpu()


@pytest.mark.gpu
@pytest.mark.parametrize("dims,R,S,dtype,occupied,t_stop", [
    ((8, 8, 8), 65, 64, torch.float32, False, 0.0),       # one tile and its wrapped halo
    ((9, 17, 5), 130, 65, torch.float32, True, 0.0),      # partial tiles, two groups
    ((33, 10, 70), 257, 128, torch.bfloat16, False, 1e-2),
    ((24, 24, 24), 1001, 256, torch.float16, True, 0.0),
    ((40, 31, 16), 511, 300, torch.float32, False, 1e-2),
    ((20, 20, 20), 3, 1, torch.float32, False, 0.0),
    ((2, 1, 2), 64, 130, torch.float32, False, 0.0),
    ((24, 20, 28), 300, 513, torch.float32, True, 0.0),   # one ray per wavefront
    ((16, 50, 16), 129, 1100, torch.bfloat16, False, 0.0),
])
def test_binned_train_step_equals_direct(dims, R, S, dtype, occupied, t_stop):
    say("bins", dims, R, S, dtype, occupied, t_stop)
    grid, o, d, gmin, pd, delta, tgt = _scene(dims, R, S, 3)
    grid, o, d, tgt = grid.to(dtype).to(DEV), o.to(DEV), d.to(DEV), tgt.to(DEV)
    bits = None
    if occupied:
        occ = torch.rand(dims, generator=torch.Generator().manual_seed(4)) < 0.3
        bits = occupancy_dilate(pack_occupancy(occ.to(DEV)), dims)
    cfg = MarchConfig(S, delta, gmin, pd, "trilinear", 0.0, t_stop)
    direct = _train(grid, o, d, tgt, cfg, bits, None)
    assert direct[3].abs().max() > 0
    whole = torch.full((1 << 26,), 0xA5, dtype=torch.uint8, device=DEV)  # its contents do not matter
    # one piece, and an offset buffer that holds a few dozen rays at a time
    for work in (whole, whole[3: 3 + (1 << 20) + 40 * 64 * S]):
        binned = _train(grid, o, d, tgt, cfg, bits, work)
        for a, b in zip(binned[:3], direct[:3]):
            assert torch.equal(a, b)
        ok, info = grad_close(binned[3], direct[3], rel=1e-5)
        say("  ", work.numel(), info)
        assert ok, info


@pytest.mark.gpu
@pytest.mark.parametrize("dims,R,S,far", [
    ((90, 97, 101), 5000, 200, False),     # 2028 tiles: two workgroups of tile ranges, the second a part of one
    ((129, 136, 130), 60000, 200, True),   # 4913 tiles, items of 512 runs, tiles of more than one item
    ((210, 201, 216), 60000, 200, False),  # 18954 tiles, most of them reached: more items than workgroups
])
def test_binned_train_step_of_many_tiles(dims, R, S, far):
    """Tile counts that take several workgroups for their ranges, whose workgroups may come in any order,
    and either number of runs per item; more items than the tile sums have workgroups.  far: a third of
    the rays cross at one place, whose tiles get thousands of runs."""
    say("bins, many tiles", dims, R, S, far)
    tiles = 1
    for n in dims:
        tiles *= (n + 7) // 8
    grid, o, d, gmin, pd, delta, tgt = _scene(dims, R, S, 13)
    if far:  # through the grid's middle
        mid = torch.tensor(gmin) + torch.tensor(dims) * (pd / 2)
        o[::3] = mid + 0.2 * torch.rand(o[::3].shape, generator=torch.Generator().manual_seed(1)) - d[::3] * (delta * S / 2)
    grid, o, d, tgt = (t.to(DEV) for t in (grid, o, d, tgt))
    cfg = MarchConfig(S, delta, gmin, pd, "trilinear")
    g, m = _grid_struct(grid, None), cfg.to_struct()
    n = _lib.lib().pxl_scatter_work_bytes(ctypes.byref(g), ctypes.byref(m), R)
    assert n > 0  # the rule takes this batch
    work = torch.full((n,), 0xA5, dtype=torch.uint8, device=DEV)
    direct, binned = (_train(grid, o, d, tgt, cfg, None, w) for w in (None, work))
    for a, b in zip(binned[:3], direct[:3]):
        assert torch.equal(a, b)
    # where a third of the rays meet, a cell sums ~10^5 FP32 terms directly: sqrt(10^5) * 2^-24 = 2e-5
    ok, info = grad_close(binned[3], direct[3], rel=4e-5 if far else 1e-5)
    # the buffer starts with the items and runs it was left with, then the runs of each tile
    head = work[(-work.data_ptr()) % 256:][:16 + 4 * tiles].view(torch.int32)
    items, runs, per_tile = int(head[0]), int(head[1]), head[4:]
    say("  ", info, "tiles", tiles, "items", items, "runs", runs)
    assert ok, info
    per_item = 512 if tiles >= 4096 else 96
    assert runs == int(per_tile.sum()) and items == int(((per_tile + per_item - 1) // per_item).sum())
    assert tiles > 1024 and tiles % 1024 != 0
    assert not far or int(per_tile.max()) > per_item
    assert dims[0] != 210 or items > 16384


@pytest.mark.gpu
@pytest.mark.parametrize("dims,R,S,dtype", [
    ((9, 17, 5), 130, 40, torch.float32),        # two rays share a group of 64 lanes
    ((24, 24, 24), 501, 128, torch.bfloat16),
    ((33, 10, 70), 257, 300, torch.float16),
    ((24, 20, 28), 300, 700, torch.float32),     # one ray per wavefront
])
def test_samples_without_a_gradient_get_no_record(dims, R, S, dtype):
    """A grid whose empty cells have alpha below zero: a sample with such cells at all corners is dropped,
    within a run too, and the gradient stays; where every sample is such a one no item is left."""
    say("bins, empty cells", dims, R, S, dtype)
    grid, o, d, gmin, pd, delta, tgt = _scene(dims, R, S, 11)
    g = torch.Generator().manual_seed(12)
    grid[..., 3][torch.rand(dims, generator=g) < 0.8] = -0.02
    grid[..., :3][torch.rand(*dims, 3, generator=g) < 0.4] = 1.5
    o, d, tgt = o.to(DEV), d.to(DEV), tgt.to(DEV)
    cfg = MarchConfig(S, delta, gmin, pd, "trilinear")
    work = torch.empty(1 << 26, dtype=torch.uint8, device=DEV)
    items = work[: 4].view(torch.int32)  # the buffer's first word counts the tile sums' items
    a, b = (_train(grid.to(dtype).to(DEV), o, d, tgt, cfg, None, w) for w in (None, work))
    assert int(items) > 0 and a[3].abs().max() > 0
    ok, info = grad_close(b[3], a[3], rel=1e-5)
    assert ok, info
    empty = grid.clone()
    empty[..., 3] = -0.5
    _, _, _, grad = _train(empty.to(dtype).to(DEV), o, d, tgt, cfg, None, work)
    assert int(items) == 0 and grad.abs().max() == 0


@pytest.mark.gpu
@pytest.mark.parametrize("S,interp", [(96, "trilinear"), (700, "trilinear"), (96, "nearest")])
def test_render_rays_backward_above_the_bin_threshold(S, interp):
    """Large enough a batch that render_rays' backward takes the bins (trilinear), against the plain
    chain's autograd; some rays with a zero upstream gradient."""
    R = (1 << 20) // S + 3
    say("render_rays backward", R, S, interp)
    grid, o, d, gmin, pd, delta, tgt = _scene((30, 22, 41), R, S, 5)
    up = torch.rand(R, 4, generator=torch.Generator().manual_seed(6)) - 0.5
    up[::7] = 0
    leaf = grid.to(DEV).requires_grad_(True)
    g, m = _grid_struct(leaf.detach(), None), MarchConfig(S, delta, gmin, pd, interp).to_struct()
    takes_bins = _lib.lib().pxl_scatter_work_bytes(ctypes.byref(g), ctypes.byref(m), R) > 0
    assert takes_bins == (interp == "trilinear")
    out = render_rays(leaf, o.to(DEV), d.to(DEV), num_samples=S, delta_step=delta, grid_min=gmin, points_distance=pd,
                      interp=interp)
    out.backward(up.to(DEV))
    ref = grid.double().requires_grad_(True)
    for a in range(0, R, 4096):
        w = plain.render(ref, o[a:a + 4096], d[a:a + 4096], num_samples=S, delta_step=delta,
                         gmin=torch.tensor(gmin), points_distance=pd, interp=interp, div_mode="reciprocal")
        (w * up[a:a + 4096].double()).sum().backward()
    ok, info = grad_close(leaf.grad.cpu(), ref.grad)
    say("  ", info)
    assert ok, info


@pytest.mark.gpu
def test_more_rays_than_one_launch():
    """2^26 + 5 rays of one and two samples: more than one launch takes, forward, backward and train step,
    binned (whose pieces the work buffer's bytes alone would not bound) and direct."""
    R, dims, pd = (1 << 26) + 5, (24, 25, 26), 0.1
    g = torch.Generator(device=DEV).manual_seed(8)
    grid = torch.rand(*dims, 4, device=DEV, generator=g) * 0.5
    o = torch.rand(R, 3, device=DEV, generator=g) * 2.2
    d = torch.zeros(R, 3, device=DEV)
    d[:, 2] = 1.0
    up = torch.rand(R, 4, device=DEV, generator=g)
    tgt = -up  # every sample's gradient is positive, so that no cell's sum cancels
    for S in (1, 2):
        say("more rays than one launch", S)
        cfg = MarchConfig(S, 0.11, (0.0, 0.0, 0.0), pd, "trilinear")
        kw = dict(num_samples=S, delta_step=0.11, grid_min=(0.0, 0.0, 0.0), points_distance=pd, interp="trilinear")
        leaf = grid.clone().requires_grad_(True)
        g_, m = _grid_struct(grid, None), cfg.to_struct()
        assert _lib.lib().pxl_scatter_work_bytes(ctypes.byref(g_), ctypes.byref(m), R) > 0
        out = render_rays(leaf, o, d, **kw)
        out.backward(up)
        parts = grid.clone().requires_grad_(True)
        for a in range(0, R, 1 << 23):
            w = render_rays(parts, o[a:a + (1 << 23)], d[a:a + (1 << 23)], **kw)
            assert torch.equal(w, out[a:a + (1 << 23)])
            w.backward(up[a:a + (1 << 23)])
        # a cell's ~10^4 records arrive in a few thousand FP32 additions of positive terms, in another
        # order: each rounds to 2^-24, sqrt(5000) * 2^-24 = 4e-6 typically and 3e-4 if all round alike
        ok, info = grad_close(leaf.grad.cpu(), parts.grad.cpu())
        assert ok, info
        grads = []
        for n in (R, R // 2):
            grad = torch.zeros_like(grid)
            for a in range(0, R, n):
                train_step(grid, grad, cfg=cfg, origins=o[a:a + n], dirs=d[a:a + n], targets=tgt[a:a + n], n_total_rays=R)
            grads.append(grad.cpu())
        ok, info = grad_close(grads[0], grads[1])
        assert ok, info


@pytest.mark.gpu
def test_binned_integer_coordinates():
    """Samples at exact integer coordinates (ceil == floor) and on the last cell, whose ceil is itself."""
    X, pd = 16, 0.25
    g = torch.Generator().manual_seed(70)
    grid = (torch.rand(X, X, X, 4, generator=g) * 0.3).to(DEV)
    o = torch.zeros(64, 3)
    o[:, 0] = -3 * pd
    o[:, 1:] = torch.randint(0, X, (64, 2), generator=g).float() * pd
    d = torch.zeros(64, 3)
    d[:, 0] = 1.0
    tgt = torch.rand(64, 4, generator=g).to(DEV)
    cfg = MarchConfig(24, pd, (0.0, 0.0, 0.0), pd, "trilinear")
    a = _train(grid, o.to(DEV), d.to(DEV), tgt, cfg, None, None)[3]
    b = _train(grid, o.to(DEV), d.to(DEV), tgt, cfg, None, torch.empty(1 << 24, dtype=torch.uint8, device=DEV))[3]
    ok, info = grad_close(b, a, rel=1e-6)
    say("bins at integer coordinates", info)
    assert ok, info


def test_scatter_work_bytes_rule():
    """No buffer for nearest lookup, small batches and grids with many more tiles than samples; at
    most 12 GiB; errors as the other entry points report them."""
    L = _lib.lib()
    g = _lib.Grid(data=0x1000, channels=4, dtype=_lib.DTYPE_F32)
    for a, n in enumerate((64, 64, 64)):
        g.dims[a] = n
    tri, near = (MarchConfig(128, 0.1, (0.0, 0.0, 0.0), 0.1, i).to_struct() for i in ("trilinear", "nearest"))
    q = lambda m, n: L.pxl_scatter_work_bytes(ctypes.byref(g), ctypes.byref(m), n)  # noqa: E731
    assert q(near, 1 << 20) == 0 and q(tri, 0) == 0 and q(tri, 100) == 0
    assert q(tri, (BIN_MIN_SAMPLES - 1) // 128) == 0 and q(tri, BIN_MIN_SAMPLES // 128) > 0
    assert 0 < q(tri, 1 << 14) < q(tri, 1 << 15) <= q(tri, 1 << 26) <= 12 << 30
    assert q(tri, -1) == _lib.PXL_E_INVALID
    g.occupancy = 0x1000
    assert q(tri, 1 << 14) == 0 and q(tri, 1 << 15) > 0
    fine = MarchConfig(128, 0.02, (0.0, 0.0, 0.0), 0.1, "trilinear").to_struct()  # five samples per cell
    assert q(fine, 1 << 17) == 0 and q(fine, 1 << 18) > 0
    g.dims[0] = 1 << 18
    assert q(tri, 1 << 14) == 0
    assert L.pxl_scatter_work_bytes(None, ctypes.byref(tri), 5) == _lib.PXL_E_INVALID


@pytest.mark.gpu
def test_binned_train_step_in_a_graph():
    """A captured step (zero, tile-binned scatter) replayed several times, with eager work and new ray
    directions between the replays, against the eager step on the same inputs."""
    S, R = 128, 1 << 13
    say("bins in a graph")
    grid, o, d, gmin, pd, delta, tgt = _scene((32, 32, 32), R, S, 9)
    grid, o, d, tgt = (t.to(DEV) for t in (grid, o, d, tgt))
    cfg = MarchConfig(S, delta, gmin, pd, "trilinear")
    g_, m = _grid_struct(grid, None), cfg.to_struct()
    assert _lib.lib().pxl_scatter_work_bytes(ctypes.byref(g_), ctypes.byref(m), R) > 0
    grad, eager = torch.zeros_like(grid), torch.zeros_like(grid)

    def step(out):
        out.zero_()
        train_step(grid, out, cfg=cfg, origins=o, dirs=d, targets=tgt)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step(grad)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step(grad)
    for i in range(4):
        d.copy_(torch.nn.functional.normalize(d + 0.01 * i, dim=1))
        step(eager)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        ok, info = grad_close(grad.cpu(), eager.cpu(), rel=1e-5)
        assert ok and eager.abs().max() > 0, (i, info)


@pytest.mark.gpu
def test_binned_train_step_asks_for_room_in_a_graph(monkeypatch):
    """The question for free memory, which only large work buffers ask, is allowed under capture."""
    asked, has_room = [], render._has_room
    monkeypatch.setattr(render, "WORK_UNASKED_BYTES", 0)
    monkeypatch.setattr(render, "_has_room", lambda n, dev: asked.append(has_room(n, dev)) or asked[-1])
    test_binned_train_step_in_a_graph()
    assert len(asked) == 6 and all(asked)
