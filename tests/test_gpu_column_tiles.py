"""Column passes at the work-group shapes that differ from length to length:
tiles of two cache lines (L = 192 in FP64), a ragged last tile (324 / 2 = 162
columns), work-groups of 64 to 320 threads whose last stage leaves lanes
idle, and the exchange of one component at a time.  Each length runs every
column tile against the float64 oracle, with the tolerances the other
operator tests hold the same transforms to."""
import numpy as np
import pytest
import torch

from oracle import convolve as ocv
from oracle.data import Domain
from tests.problems import psf_windows

pytestmark = pytest.mark.gpu

TOL = {torch.float64: 1e-12, torch.float32: 2e-6}


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("H,n,m,L", [(8, 2, 4, 16),       # 8 stored columns, one tile
                                     (32, 2, 8, 48),      # 64 threads, 24 columns
                                     (128, 4, 16, 96),    # 128 threads
                                     (128, 2, 32, 192),   # split exchange; FP64: 16 columns
                                     (256, 2, 32, 320),   # 192 threads in FP64
                                     (303, 3, 61, 324),   # 320 threads, 162 columns
                                     (304, 2, 64, 432),   # 27-point butterflies
                                     (256, 2, 128, 512)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_column_tiles_vs_oracle(ja, H, n, m, L, dtype):
    E = 2
    rng = np.random.default_rng(L)
    win = psf_windows(rng, n, E, 2 * (H // n))
    op = ja.LinpatchOperator((E, H, H), n, m, dtype=dtype)
    assert op.L == L
    op.set_kernel(win, layout="window")
    dom = Domain((E, H, H), (1.0, 1.0, 1.0))
    x, g = rng.random((E, H, H)), rng.normal(size=(E, H, H))
    want_y = ocv.linpatch_convolve_window(x, dom, win, n, m)
    want_g = ocv.linpatch_adjoint_window(g, dom, win, n, m)
    for div in (1, 2, 4):
        op.set_tile(div)
        y = op.forward(torch.as_tensor(x, dtype=dtype, device="cuda"))
        gx = op.adjoint(torch.as_tensor(g, dtype=dtype, device="cuda"))
        assert _rel(y.double().cpu().numpy(), want_y) <= TOL[dtype], f"forward, tile 1/{div}"
        assert _rel(gx.double().cpu().numpy(), want_g) <= TOL[dtype], f"adjoint, tile 1/{div}"
