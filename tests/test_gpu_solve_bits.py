"""Conjugate-gradient steps in FP32 at a stiff observation, where a solution
that is not converged depends on the last bits of the metric products: a fixed
number of steps gives what it gave when these values were recorded."""
import numpy as np
import pytest
import torch

from tests.problems import psf_windows

pytestmark = pytest.mark.gpu

STEPS = 8
# ((N, H, n, m), seed): projections of the two solutions (_projections).  The
# transform lengths are 192, 128, 96 and 432 (fold mode), the GP grids in LDS
# and in registers; the seeds are such that a change of rounding in the metric
# (9e-8 of a product) moves a solution by 4e-4 to 4e-2.
RECORDED = {
    ((256, 256, 4, 32), 9): [
     [1.4106882, 0.2445107, 0.2223044, -1.8768936,
      0.0864565, -0.5802096, -1.0096189, -0.0787435],
     [0.2184153, -0.1464894, 1.6631211, 0.9201127,
      -0.8372042, -0.8644770, 0.7656590, -0.1670485]],
    ((256, 256, 6, 22), 4): [
     [0.5846452, 0.5754224, -0.3097118, 0.7690196,
      -0.6608368, -0.7177281, 0.4543450, 1.0627428],
     [1.4725427, 0.8619865, -1.1952904, -1.5048821,
      -0.2916560, -0.4368726, 0.9740096, -1.0794798]],
    ((128, 128, 4, 16), 2): [
     [0.9868397, -1.7035447, 0.0138772, 0.5615530,
      1.2569803, -0.0825311, 0.6463213, 2.6908127],
     [0.2943926, 0.1505949, -1.1034210, 1.3151752,
      -0.1774842, -0.0329464, -0.1770445, 0.9197169]],
    ((567, 512, 5, 30), 3): [
     [1.1902376, -0.2957725, -0.0497932, 0.1979202,
      -1.6720160, 0.3044083, 1.1057887, -0.7829287],
     [-0.1510155, 1.2025901, -0.5423230, -1.4958605,
      -0.3012741, -0.9017275, -0.2664182, -1.9966146]],
}


def _solve(ja, N, H, n, m, seed, samples=2):
    rng = np.random.default_rng(seed)
    k = np.fft.fftfreq(N)
    amp = k[:, None] ** 2 + k[None, :] ** 2
    amp[0, 0] = np.inf
    amp = 1.0 / amp
    amp /= np.sqrt((amp ** 2).sum())
    win = psf_windows(rng, n, 1, 2 * (H // n))
    expo = np.broadcast_to(np.linspace(5e2, 2e3, H), (1, 1, H, H)).copy()
    keep = rng.random((1, 1, H, H)) >= 0.05
    counts = np.where(keep, rng.integers(0, 300, (1, 1, H, H)), -1)
    xi = rng.standard_normal((N, N))
    b = rng.standard_normal((samples, N, N))
    dev = lambda a, dt=torch.float32: torch.as_tensor(a, dtype=dt, device="cuda")  # noqa: E731
    sky = ja.CorrelatedFieldSky(N, (H, H), dev(amp), None, zm=-2.0, mu=0.0, dnu=np.zeros(1),
                                dtype=torch.float32)
    op = ja.LinpatchOperator((1, H, H), n, m, n_modules=1, dtype=torch.float32)
    op.set_kernel(dev(win), layout="window")
    model = ja.XrayModel(sky, op, 1.0, dev(expo * keep), dev(counts, torch.int32),
                         max_samples=samples)
    model.nll_and_grad(dev(xi))
    model.reserve_solver()
    return model.metric_solve(dev(b), None, maxiter=STEPS)[0][0]


def _projections(x):
    """Dot products of every solution with eight fixed fields of unit variance,
    over its norm."""
    rng = np.random.default_rng(0)
    w = rng.standard_normal((8, x[0].numel()))
    v = x.double().cpu().numpy().reshape(len(x), -1)
    return v @ w.T / np.linalg.norm(v, axis=1, keepdims=True)


@pytest.mark.parametrize("case", RECORDED)
def test_steps_are_the_recorded_ones(ja, case):
    geometry, seed = case
    got = _projections(_solve(ja, *geometry, seed))
    assert np.abs(got - np.array(RECORDED[case])).max() <= 2e-5
