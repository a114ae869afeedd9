"""The end of a training step: Adam on a pooled grid's gradient in one pass (the bits of the pooling
backward followed by Adam) and the loss values in one launch."""
import math

import pytest
import torch

from plenoxels_amd.grid_functions import pool_backward_
from plenoxels_amd.optim import adam_pooled_step_, adam_step_
from plenoxels_amd.render import LossTerms, beta_term_zero
from util import say

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
