"""The end of a training step: Adam on a pooled grid's gradient in one pass (the bits of the pooling
backward followed by Adam) and the loss values in one launch."""
import math

import pytest
import torch

from plenoxels_amd.grid_functions import pool_backward_
from plenoxels_amd.optim import adam_pooled_step_, adam_step_
from plenoxels_amd.render import LossTerms, beta_term_zero
from plenoxels_amd.train import Trainer
from util import random_cameras, say

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("dims,k,s", [((3, 3, 3), 3, 1), ((7, 9, 64), 5, 1), ((20, 17, 33), 9, 2), ((12, 30, 65), 11, 2),
                                      ((40, 31, 29), 25, 6), ((5, 5, 300), 5, 7)])
@pytest.mark.parametrize("half", [None, torch.bfloat16, torch.float16])
def test_adam_pooled_equals_pool_backward_then_adam(dims, k, s, half):
    say("adam pooled", dims, k, s, half)
    g = torch.Generator(device=DEV).manual_seed(k)
    rnd = lambda *shape: torch.randn(*shape, device=DEV, generator=g)  # noqa: E731
    out_dims = [(n - k) // s + 1 for n in dims]
    go, p, m, v, a = rnd(*out_dims, 4), rnd(*dims, 4), rnd(*dims, 4), rnd(*dims, 4).abs(), rnd(*dims, 4).abs()
    want = [t.clone() for t in (p, m, v, a)]
    got = [t.clone() for t in (p, m, v, a)]
    halves = [None if half is None else torch.zeros(*dims, 4, dtype=half, device=DEV) for _ in range(2)]
    grad = torch.empty(*dims, 4, device=DEV)
    pool_backward_(go, dims, k, s, grad, accumulate=False)
    adam_step_(want[0], grad, want[1], want[2], 7, lr=0.03, grad_abs=want[3], half_out=halves[0])
    adam_pooled_step_(got[0], go, k, s, got[1], got[2], 7, lr=0.03, grad_abs=got[3], half_out=halves[1])
    for x, y in zip(want, got):
        assert torch.equal(x, y)
    assert half is None or torch.equal(*halves)


@pytest.mark.parametrize("interp,step", [("nearest", 200), ("trilinear", 226)])  # receptive fields 13 and 3
def test_trainer_grad_after_a_pooled_step(interp, step):
    """Trainer.grad after a pooled step is that step's gradient to the full grid: |grad| is what the
    step added to grad_abs.  A full-grid step after it starts from a clean buffer."""
    say("trainer grad", interp, step)
    g = torch.Generator().manual_seed(step)
    c2w = random_cameras(4, 3)
    kw = dict(gridsize=(24, 20, 22), points_distance=0.1, number_of_rays=60, num_samples=70, delta_step=0.05, lr=0.01,
              tv=1e-3, beta=1e-3, interp=interp, init_grid=torch.rand(24, 20, 22, 4, generator=g) * 0.3)
    uv = torch.rand(4, 60, 2, generator=g)
    imgs = torch.rand(4, 16, 16, 4, generator=g)
    a, b = (Trainer(imgs, c2w, 0.7, uniforms_fn=lambda i: uv, **kw) for _ in range(2))
    a.step(step)
    assert a.grad.abs().max() > 0 and torch.equal(a.grad.abs(), a.grad_abs)
    assert a.grad is a.grad
    buffer = torch.ones_like(a.grad)
    a.grad = buffer  # another buffer may take its place, whatever it holds
    assert a.grad is buffer
    # reading it changes nothing that follows
    b.step(step)
    for _ in range(2):
        a.step(230), b.step(230)
        assert a.grad.abs().max() == 0  # the fused TV + Adam pass leaves it zero
    # the scatters' order differs, and a first Adam step divides a gradient by its own size, so a cell whose
    # terms cancel may move differently; a gradient left in the buffer would move most cells by ~0.01
    assert (a.grid - b.grid).abs().mean() < 1e-5


@pytest.mark.parametrize("n", [1, 2, 255, 16385, 100003, (1 << 19) + 7])
@pytest.mark.parametrize("tv,beta", [(False, False), (True, False), (False, True), (True, True)])
def test_loss_terms(n, tv, beta):
    say("loss terms", n, tv, beta)
    g = torch.Generator().manual_seed(n)
    sq, bs = torch.rand(n, generator=g), torch.randn(n, generator=g)
    tvs = torch.tensor([12.75], dtype=torch.float64, device=DEV)
    terms = LossTerms(DEV)
    S, rays = 64, max(n, 1)
    for _ in range(3):  # the work buffer serves call after call
        got = terms(sq.to(DEV), rays, tv_sumsq=tvs if tv else None, tv_weight=1e-3, ray_beta=bs.to(DEV) if beta else None,
                    beta=5e-3, n_samples=rays * S).tolist()
        want = [math.fsum(sq.tolist()) / (4 * rays), 1e-3 * math.sqrt(12.75) if tv else 0.0,
                5e-3 * (math.fsum(bs.tolist()) + rays * S * beta_term_zero()) / (rays * S) if beta else 0.0]
        # float64 sums rounded once to float32; the total rounds twice more
        for a, b in zip(got, want):
            assert abs(a - b) <= 2.0 ** -23 * abs(b) + 1e-300
        assert abs(got[3] - sum(want)) <= 3 * 2.0 ** -23 * sum(abs(w) for w in want) + 1e-300
