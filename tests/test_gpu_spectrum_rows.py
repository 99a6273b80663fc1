"""The column pass's row-strided accesses at their edges: windows that leave
the image on either side, spectra whose half length does not fill the last
column tile, fold mode, and rows outside a window that are not finite."""
import numpy as np
import pytest
import torch

from oracle import convolve as cv
from oracle.data import Domain as ODomain
from tests.problems import psf_windows

pytestmark = pytest.mark.gpu

# (H, n, m): half lengths of 12, 24 (partial and full tiles of 16 and 8),
# 162 (ten tiles and a remainder), 192, 256; fold mode (w + 2m = 22, 86, 332);
# odd strides with a clamped last window, images larger than n strides.
GEOMS = [(16, 2, 4), (48, 4, 12), (49, 4, 11), (34, 4, 3), (90, 4, 21), (307, 3, 60),
         (257, 2, 128), (386, 3, 64), (306, 3, 64)]


@pytest.mark.parametrize("H,n,m", GEOMS)
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_both_directions_match_oracle(ja, H, n, m, dtype):
    E = 2
    rng = np.random.default_rng(H + n + m)
    win = psf_windows(rng, n, E, 2 * (H // n))
    x, g = rng.normal(size=(2, E, H, H))
    dom = ODomain((E, H, H), (1.0, 1.0, 1.0))
    op = ja.LinpatchOperator((E, H, H), n, m, dtype=dtype)
    op.set_kernel(win, layout="window")
    tol = 1e-12 if dtype == torch.float64 else 2e-6  # as for the other geometries
    for got, want in ((op.forward(torch.as_tensor(x, device="cuda")),
                       cv.linpatch_convolve_window(x, dom, win, n, m)),
                      (op.adjoint(torch.as_tensor(g, device="cuda")),
                       cv.linpatch_adjoint_window(g, dom, win, n, m))):
        err = np.linalg.norm(got.double().cpu().numpy() - want) / np.linalg.norm(want)
        assert err <= tol


@pytest.mark.parametrize("H,n,m", [(128, 4, 16), (256, 4, 32), (306, 3, 60), (306, 3, 64)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_other_windows_rows_do_not_enter(ja, H, n, m, dtype):
    """A NaN in the last row spoils the windows that hold it and no other:
    the rows next to a window read as zero, whatever they hold."""
    d = H // n
    win = psf_windows(np.random.default_rng(1), n, 1, 2 * d)
    op = ja.LinpatchOperator((1, H, H), n, m, dtype=dtype)
    op.set_kernel(win, layout="window")
    x = torch.ones((1, H, H), dtype=dtype, device="cuda")
    x[0, -1] = float("nan")
    hit = min(i for i in range(n) if i * d - d // 2 + 2 * d >= H)
    clean = hit * d - d // 2
    assert torch.isfinite(op.forward(x)[0, :clean - m]).all()
    # adjoint: windows with their margins
    hit = min(i for i in range(n) if i * d - d // 2 + 2 * d + m >= H)
    assert torch.isfinite(op.adjoint(x)[0, :hit * d - d // 2]).all()
