"""Checks of the Python layer that need no GPU: what a kernel would read or write out of range, or as
another type, is refused before any pointer leaves Python, and a work buffer is asked for only
where there is room."""
import ctypes

import pytest
import torch

from plenoxels_amd import MarchConfig, _lib, render
from plenoxels_amd.optim import adam_pooled_step_
from plenoxels_amd.render import LossTerms, alpha_occupancy


def test_loss_terms_rejects_what_its_kernel_would_misread():
    terms = LossTerms("cpu")
    sq, bs, tv = torch.zeros(64), torch.zeros(64), torch.zeros(1, dtype=torch.float64)
    for bad in (sq.double(), sq.reshape(8, 8), torch.zeros(128)[::2], sq.to("meta")):
        with pytest.raises(ValueError, match="ray_sq_err must be"):
            terms(bad, 64)
        with pytest.raises(ValueError, match="ray_beta must be"):
            terms(sq, 64, ray_beta=bad, beta=1.0, n_samples=64)
    for n in (63, 65, 0):
        with pytest.raises(ValueError, match="length"):
            terms(sq, 64, ray_beta=torch.zeros(n), beta=1.0, n_samples=64)
    for bad in (tv.float(), torch.zeros(2, dtype=torch.float64), tv.to("meta")):
        with pytest.raises(ValueError, match="tv_sumsq must be"):
            terms(sq, 64, tv_sumsq=bad, tv_weight=1.0)
    with pytest.raises(ValueError, match="HIP device"):
        terms(sq, 64, tv_sumsq=tv, tv_weight=1.0, ray_beta=bs, beta=1.0, n_samples=64)


def test_adam_pooled_step_rejects_arrays_of_other_shapes():
    dims, k, s = (8, 9, 10), 3, 2
    p, m, v, a = (torch.zeros(*dims, 4) for _ in range(4))
    go = torch.zeros(3, 4, 4, 4)
    for bad in (go[:2], go[:, :3], torch.zeros(4, 4, 3, 4), torch.zeros(3, 4, 4), go.to("meta")):
        with pytest.raises(ValueError, match="grad_out must"):
            adam_pooled_step_(p, bad, k, s, m, v, 1, lr=1.0, grad_abs=a)
    for bad in (m[:7], m.double(), torch.zeros(8, 9, 20, 4)[:, :, ::2], m.to("meta")):
        with pytest.raises(ValueError, match="exp_avg must"):
            adam_pooled_step_(p, go, k, s, bad, v, 1, lr=1.0)
        with pytest.raises(ValueError, match="exp_avg_sq must"):
            adam_pooled_step_(p, go, k, s, m, bad, 1, lr=1.0)
        with pytest.raises(ValueError, match="grad_abs must"):
            adam_pooled_step_(p, go, k, s, m, v, 1, lr=1.0, grad_abs=bad)
    with pytest.raises(ValueError, match="half_out must"):
        adam_pooled_step_(p, go, k, s, m, v, 1, lr=1.0, half_out=torch.zeros(7, 9, 10, 4, dtype=torch.bfloat16))
    with pytest.raises(ValueError, match="average pooling needs"):
        adam_pooled_step_(p, go, 9, s, m, v, 1, lr=1.0)


def test_alpha_occupancy_rejects_a_tv_sum_of_another_type_or_place():
    grid = torch.zeros(4, 4, 4, 4)
    for bad in (torch.zeros(1), torch.zeros(2, dtype=torch.float64), torch.zeros(0, dtype=torch.float64),
                torch.zeros(1, dtype=torch.float64, device="meta")):
        with pytest.raises(ValueError, match="tv_sumsq must be"):
            alpha_occupancy(grid, "nearest", tv_sumsq=bad)


@pytest.mark.parametrize("free,reserved,allocated,fraction,capturing,want", [
    (1 << 40, 0, 0, 1.0, False, 1),                # room on the device
    (1 << 20, 1 << 40, 0, 1.0, False, 1),          # room in torch's cache
    (1 << 20, 5 << 30, 5 << 30, 1.0, False, 0),    # no room: nothing is asked for
    (3 << 30, 5 << 30, 5 << 30, 1.0, False, 4),    # room for a quarter
    (1 << 40, 5 << 30, 5 << 30, 0.005, False, 0),  # the process may not take what is free
    (1 << 40, 0, 0, 0.5, False, 1),
    (1 << 20, 1 << 40, 0, 1.0, True, 0),           # a capture does not draw on the cache
    (1 << 40, 0, 0, 1.0, True, 1),
])
def test_scatter_work_asks_only_for_what_there_is_room_for(monkeypatch, free, reserved, allocated, fraction, capturing,
                                                          want):
    g = _lib.Grid(data=0x1000, channels=4, dtype=_lib.DTYPE_F32)
    g.dims[:] = (256, 256, 256)
    m = MarchConfig(512, 0.1, (0.0, 0.0, 0.0), 0.1, "trilinear").to_struct()
    n = _lib.lib().pxl_scatter_work_bytes(ctypes.byref(g), ctypes.byref(m), 1 << 19)
    assert n > 8 << 30
    asked = []
    monkeypatch.setattr(torch, "empty", lambda size, **kw: asked.append(size) or "buffer")
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda dev: (free, 288 << 30))
    monkeypatch.setattr(torch.cuda, "memory_reserved", lambda dev: reserved)
    monkeypatch.setattr(torch.cuda, "memory_allocated", lambda dev: allocated)
    monkeypatch.setattr(torch.cuda, "get_per_process_memory_fraction", lambda dev: fraction)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing)
    work = render._scatter_work(g, m, 1 << 19, torch.device("cuda:0"))
    assert asked == {0: [], 1: [n], 4: [n // 4]}[want] and (work is None) == (want == 0)
