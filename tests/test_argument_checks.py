"""Argument checks of the Python layer that need no GPU: what a kernel would read or write out of
range, or as another type, is refused before any pointer leaves Python."""
import pytest
import torch

from plenoxels_amd.render import LossTerms


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
