"""The sampled KL's sums on the device (jubik_model_kl_grad) against the same
sums as array operations, which inputs of other dtypes, layouts or shapes
still take: both grids whose fields allow 16-byte accesses and odd ones, one
and two fields, misaligned views, and the smallest and largest batch.
Tolerances: the prior energy and the mean are sums in double (rounding of the
last bit in the model's dtype); the NLL is the same kernel's."""
import numpy as np
import pytest
import torch

from tests.problems import make_problem, to_product

from jubik_amd import kl  # importable once tests.problems has loaded the package

pytestmark = pytest.mark.gpu


def _arrays(model, xi, S, dtype, seed, offset=0):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    out = []
    for x in xi:
        if x is None:
            out += [None, None]
            continue
        n = x.size
        buf = torch.empty(n + offset, dtype=dtype, device="cuda")[offset:].view(x.shape)
        buf.copy_(torch.as_tensor(x))
        d = torch.empty(S * n + offset, dtype=dtype, device="cuda")[offset:].view((S,) + x.shape)
        d.copy_(0.1 * torch.randn((S,) + x.shape, generator=gen, device="cuda"))
        out += [buf, d]
    return out


@pytest.mark.parametrize("E,N,H", [(1, 64, 64), (2, 64, 60), (2, 567, 62)])
@pytest.mark.parametrize("S,offset", [(1, 0), (3, 0), (4, 1)])
@pytest.mark.parametrize("dtype,eps", [(torch.float32, 2.0 ** -23), (torch.float64, 2.0 ** -52)])
def test_fused_kl_equals_array_operations(ja, E, N, H, S, offset, dtype, eps, monkeypatch):
    prob, xi = make_problem(H=H, n=4, margin=8, E=E, M=1, seed=E + N + S, N=N)
    model = to_product(ja, prob, dtype, max_samples=4)
    xr, dr, xa, da = _arrays(model, xi, S, dtype, seed=S, offset=offset)
    assert kl._on_device(model, xr, xa, dr, da)
    value, (g_r, g_a) = ja.kl_value_and_grad(model, xr, xa, dr, da)
    monkeypatch.setattr(kl, "_on_device", lambda *a: False)
    want, (w_r, w_a) = ja.kl_value_and_grad(model, xr, xa, dr, da)
    assert abs(value - want) <= 1e-13 * abs(want)
    for g, w in ((g_r, w_r), (g_a, w_a)):
        assert (g is None) == (w is None)
        if g is not None:
            assert g.dtype == dtype and g.shape == w.shape
            # each side rounds a double once; the doubles differ by the rounding
            # of a few sums whose terms are bounded by max|w| + max|position|
            most = float(w.abs().max()) + 10.0
            assert float(((g - w).abs() - 2 * eps * w.abs()).max()) <= 8 * 2.0 ** -52 * most


def test_other_inputs_take_the_array_operations(ja):
    prob, xi = make_problem(H=64, n=4, margin=8, E=2, M=1, seed=3)
    model = to_product(ja, prob, torch.float32, max_samples=3)
    xr, dr, xa, da = _arrays(model, xi, 3, torch.float32, seed=1)
    want, (w_r, _) = ja.kl_value_and_grad(model, xr, xa, dr, da)
    others = [(xr.double(), xa, dr, da),                      # another dtype
              (xr.t().contiguous().t(), xa, dr, da),          # another order
              (xr[None], xa, dr, da)]                         # broadcasting shape
    for args in others:
        assert not kl._on_device(model, *args)
    for args in others[:2]:
        value, (g_r, _) = ja.kl_value_and_grad(model, *args)
        assert abs(value - want) <= 1e-6 * abs(want)
        np.testing.assert_allclose(g_r.cpu().numpy(), w_r.cpu().numpy(), rtol=1e-4, atol=1e-3)
