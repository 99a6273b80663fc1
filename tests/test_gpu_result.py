"""The host-side report of a gradient evaluation (jubik_model_result): the
NLL values and domain counts that the kernels write to page-locked memory
equal the device results, for one position, for the smallest and largest
batch, and for a replayed graph."""
import ctypes

import numpy as np
import pytest
import torch

from tests.problems import make_problem, to_product

pytestmark = pytest.mark.gpu


def _result(model, S):
    from jubik_amd import _device, _lib
    nll, counts = (ctypes.c_double * S)(), (ctypes.c_int64 * S)()
    _lib.call("jubik_model_result", model._model, nll, counts, _device.stream())
    return list(nll), list(counts)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("S", [1, 2, 5])
def test_report_equals_device_values(ja, S, dtype):
    prob, (xr, xa) = make_problem(H=64, n=4, margin=8, E=2, M=1, seed=5)
    model = to_product(ja, prob, dtype, max_samples=5)
    dev = lambda a: torch.as_tensor(a, dtype=dtype, device="cuda")  # noqa: E731
    nll, _, _ = model.nll_and_grad_device(dev(xr), dev(xa))
    got, counts = _result(model, 1)
    assert got == [float(nll.item())] and counts == [0]
    steps = [0.01 * k for k in range(S)]
    pr = torch.stack([dev(xr) + s for s in steps])
    pa = torch.stack([dev(xa) - s for s in steps])
    vals, _, _ = model.nll_and_grad_batch(pr, pa)
    assert vals.dtype == np.float64 and vals.shape == (S,)
    for k in range(S):
        one, _, _ = model.nll_and_grad_device(pr[k].contiguous(), pa[k].contiguous())
        assert vals[k] == float(one.item())


def test_report_after_graph_replays(ja):
    prob, (xr, xa) = make_problem(H=64, n=4, margin=8, E=2, M=1, seed=6)
    model = to_product(ja, prob, torch.float32)
    graph = model.capture_grad()
    for k in range(3):
        graph.xi_ref.copy_(torch.as_tensor(xr + 0.01 * k))
        graph.xi_alpha.copy_(torch.as_tensor(xa))
        graph.launch()
        got, _ = _result(model, 1)
        assert got == [float(graph.nll.item())]
        eager, _, _ = model.nll_and_grad(graph.xi_ref, graph.xi_alpha)
        assert eager == got[0]


def test_domain_counts_in_the_report(ja):
    prob, (xr, xa) = make_problem(H=64, n=4, margin=8, E=2, M=1, seed=7)
    model = to_product(ja, prob, torch.float32)
    model.exposure[0, 1, 10, 5:9] = 0.0
    model.counts[0, 1, 10, 5:9] = 3  # read out without exposure
    model.nll_and_grad_device(torch.as_tensor(xr, device="cuda"),
                              torch.as_tensor(xa, device="cuda"))
    assert list(model.check_domain(raise_error=False)) == [4]
    with pytest.raises(FloatingPointError):
        _result(model, 1)
