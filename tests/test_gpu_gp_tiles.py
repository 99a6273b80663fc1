"""The GP column pass at both tile widths: every compiled grid, crops that end
inside a tile, with and without the spectral index, real and complex cotangent
planes, against numpy in float64."""
import numpy as np
import pytest
import torch

from tests.problems import make_problem, to_product

pytestmark = pytest.mark.gpu

GRIDS = [16, 32, 64, 128, 256, 512, 567, 768, 1024, 1134, 2048]


def _ht(u):
    f = np.fft.fft2(u)
    return f.real + f.imag


@pytest.mark.parametrize("N", GRIDS)
@pytest.mark.parametrize("E", [1, 3])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_sky_and_transpose_match_numpy(ja, N, E, dtype):
    rng = np.random.default_rng(N + E)
    H = N - N // 9  # ends inside a tile
    k = np.fft.fftfreq(N)
    amp = 1.0 / (1.0 + (16.0 * np.hypot(k[:, None], k[None, :])) ** 2)
    amp /= np.sqrt((amp ** 2).sum())
    amp2 = 0.5 * amp if E > 1 else None
    xi, xa = rng.standard_normal((2, N, N))
    dnu = np.linspace(-0.5, 0.7, E)
    sky = ja.CorrelatedFieldSky(N, (H, H), amp, amp2, zm=-1.0, mu=-0.3 if E > 1 else 0.0, dnu=dnu,
                                dtype=dtype)
    t = lambda a: torch.as_tensor(a, dtype=dtype, device="cuda")  # noqa: E731
    s = sky(t(xi), t(xa) if E > 1 else None)
    ls = _ht(amp * xi)[None] - 1.0
    if E > 1:
        ls = ls + (_ht(amp2 * xa) - 0.3)[None] * dnu[:, None, None]
    want = np.exp(ls)[:, :H, :H]
    # log2(N^2) rounded stages on values of order one, and the exponential
    eps = 4 * np.log2(N * N) * torch.finfo(dtype).eps
    got = s.double().cpu().numpy()
    assert np.linalg.norm(got - want) <= eps * np.linalg.norm(want)
    y = rng.standard_normal((E, H, H))
    g_r, g_a = sky.vjp(s, t(y))
    u = np.zeros((E, N, N))
    u[:, :H, :H] = got * y
    for g, a, v in ((g_r, amp, u.sum(0)), (g_a, amp2, (u * dnu[:, None, None]).sum(0))):
        if g is None:
            continue
        want = a * _ht(v)
        assert np.linalg.norm(g.double().cpu().numpy() - want) <= eps * np.linalg.norm(want)


@pytest.mark.parametrize("dtype,tol", [(torch.float64, 1e-12), (torch.float32, 1e-5)])
def test_wide_tiles_of_a_batch_match_one_sample(ja, dtype, tol):
    """32 samples on a 64 grid take wide tiles, one sample narrow ones."""
    prob, xi = make_problem(H=64, n=4, margin=8, E=2, M=1, seed=3)
    S = 32
    one = to_product(ja, prob, dtype=dtype)
    many = to_product(ja, prob, dtype=dtype, max_samples=S)
    rng = np.random.default_rng(5)
    xs = [torch.as_tensor(v[None] + 0.1 * rng.standard_normal((S,) + v.shape), dtype=dtype,
                          device="cuda") for v in xi]
    nll, g_r, g_a = many.nll_and_grad_batch(*xs)
    for i in (0, 17, S - 1):
        n1, r1, a1 = one.nll_and_grad(xs[0][i].contiguous(), xs[1][i].contiguous())
        assert abs(nll[i] - n1) <= tol * abs(n1)
        for a, b in ((g_r[i], r1), (g_a[i], a1)):
            assert float((a - b).double().norm()) <= tol * float(b.double().norm())
