"""What jubik_model_result reports follows the evaluation that ran last, by a
call or by the launch of a graph, whatever ran or was captured before it."""
import ctypes
import math

import pytest
import torch

from tests.problems import make_problem, to_product

pytestmark = pytest.mark.gpu

MOST = 5


def _model(ja, seed):
    prob, (xr, xa) = make_problem(H=64, n=4, margin=8, E=2, M=1, seed=seed)
    model = to_product(ja, prob, torch.float32, max_samples=MOST)
    dev = lambda a: torch.as_tensor(a, dtype=torch.float32, device="cuda")  # noqa: E731
    return model, dev(xr), dev(xa)


def _batch(xr, xa, S):
    steps = [0.01 * k for k in range(S)]
    return (torch.stack([xr + s for s in steps]), torch.stack([xa - s for s in steps]))


def _result(model):
    """The values written, of MOST buffers filled with NaN."""
    from jubik_amd import _device, _lib
    nll = (ctypes.c_double * MOST)(*[math.nan] * MOST)
    _lib.call("jubik_model_result", model._model, nll, None, _device.stream())
    return [v for v in nll if not math.isnan(v)]


def test_one_sample_graph_after_a_larger_batch(ja):
    model, xr, xa = _model(ja, 11)
    graph = model.capture_grad()
    graph.xi_ref.copy_(xr)
    graph.xi_alpha.copy_(xa)
    model.nll_and_grad_batch(*_batch(xr, xa, MOST))
    graph.launch()
    assert _result(model) == [float(graph.nll.item())]


def test_batch_graph_after_one_evaluation(ja):
    model, xr, xa = _model(ja, 12)
    graph = model.capture_grad(3)
    pr, pa = _batch(xr, xa, 3)
    graph.xi_ref.copy_(pr)
    graph.xi_alpha.copy_(pa)
    model.nll_and_grad(xr, xa)
    for _ in range(3):
        graph.launch()
        assert _result(model) == graph.nll.tolist()
        model.nll_and_grad(xr, xa)


def test_domain_counts_of_a_batch_graph(ja):
    model, xr, xa = _model(ja, 13)
    model.exposure[0, 1, 10, 5:9] = 0.0
    model.counts[0, 1, 10, 5:9] = 3  # read out without exposure
    graph = model.capture_grad(3)
    pr, pa = _batch(xr, xa, 3)
    graph.xi_ref.copy_(pr)
    graph.xi_alpha.copy_(pa)
    model.nll_and_grad_device(xr, xa)
    graph.launch()
    assert list(model.check_domain(raise_error=False))[:3] == [4, 4, 4]


def test_capture_evaluates_nothing(ja):
    model, xr, xa = _model(ja, 14)
    graph = model.capture_grad(2)
    with pytest.raises(RuntimeError, match="no gradient evaluation"):
        _result(model)
    model.nll_and_grad_batch(*_batch(xr, xa, 3))
    other = model.capture_grad()
    assert len(_result(model)) == 3
    del graph, other
