"""Overlap passes at the widest rows, sixteen output columns per thread (W
over 2048), and on skies that are not square, where only one axis has a clamped
last start."""
import numpy as np
import pytest
import torch

from oracle import convolve as cv
from oracle.data import Domain as ODomain
from tests.problems import psf_windows

pytestmark = pytest.mark.gpu


# strides 32 (even: no start is clamped) and 31 (n d clamps the last start,
# n d + 1 does not)
@pytest.mark.parametrize("H,W,n,m", [(2048, 2050, 64, 16), (155, 156, 5, 17), (156, 155, 5, 17),
                                     (279, 280, 9, 17), (280, 279, 9, 17)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_wide_and_oblong_skies_match_oracle(ja, H, W, n, m, dtype):
    rng = np.random.default_rng(H + W)
    win = psf_windows(rng, n, 1, 2 * (H // n))
    x, g = rng.normal(size=(2, 1, H, W))
    dom = ODomain((1, H, W), (1.0, 1.0, 1.0))
    op = ja.LinpatchOperator((1, H, W), n, m, dtype=dtype)
    op.set_kernel(win, layout="window")
    tol = 1e-12 if dtype == torch.float64 else 2e-6  # as for the other geometries
    for got, want in ((op.forward(torch.as_tensor(x, device="cuda")),
                       cv.linpatch_convolve_window(x, dom, win, n, m)),
                      (op.adjoint(torch.as_tensor(g, device="cuda")),
                       cv.linpatch_adjoint_window(g, dom, win, n, m))):
        err = np.linalg.norm(got.double().cpu().numpy() - want) / np.linalg.norm(want)
        assert err <= tol
