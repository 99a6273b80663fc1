"""Output columns of the overlap passes: widths on both sides of one, two and
four columns per thread, more patch columns than one batch of pairs holds, and
windows that meet a row up to four times, with and without a clamped last
start."""
import numpy as np
import pytest
import torch

from oracle import convolve as cv
from oracle.data import Domain as ODomain
from tests.problems import psf_windows

pytestmark = pytest.mark.gpu


# (H, n, m): widths 255, 257, 511, 513, 1025 (odd strides among them, n d = H
# clamps the last start); n of 9 and 16 (two batches); margins over d / 2
GEOMS = [(255, 5, 8), (257, 4, 32), (511, 7, 21), (513, 9, 28), (1025, 5, 11), (144, 16, 5),
         (153, 9, 15), (256, 6, 22), (200, 8, 23)]


@pytest.mark.parametrize("H,n,m", GEOMS)
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_widths_and_batches_match_oracle(ja, H, n, m, dtype):
    rng = np.random.default_rng(H * n + m)
    win = psf_windows(rng, n, 1, 2 * (H // n))
    x, g = rng.normal(size=(2, 1, H, H))
    dom = ODomain((1, H, H), (1.0, 1.0, 1.0))
    op = ja.LinpatchOperator((1, H, H), n, m, dtype=dtype)
    op.set_kernel(win, layout="window")
    tol = 1e-12 if dtype == torch.float64 else 2e-6  # as for the other geometries
    for got, want in ((op.forward(torch.as_tensor(x, device="cuda")),
                       cv.linpatch_convolve_window(x, dom, win, n, m)),
                      (op.adjoint(torch.as_tensor(g, device="cuda")),
                       cv.linpatch_adjoint_window(g, dom, win, n, m))):
        err = np.linalg.norm(got.double().cpu().numpy() - want) / np.linalg.norm(want)
        assert err <= tol
