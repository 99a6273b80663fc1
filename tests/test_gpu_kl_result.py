"""jubik_model_kl_result belongs to the sampled KL that ran last, and is refused
once the model evaluated anything else."""
import ctypes

import pytest
import torch

from tests.problems import make_problem, to_product

pytestmark = pytest.mark.gpu


def _kl_result(model, S):
    from jubik_amd import _device, _lib
    nll, prior = (ctypes.c_double * S)(), ctypes.c_double()
    _lib.call("jubik_model_kl_result", model._model, nll, ctypes.byref(prior), _device.stream())
    return list(nll), prior.value


def test_kl_result_needs_the_kl_last(ja):
    prob, xi = make_problem(H=64, n=4, margin=8, E=2, M=1, seed=15)
    model = to_product(ja, prob, torch.float32, max_samples=2)
    xr, xa = (torch.as_tensor(a, dtype=torch.float32, device="cuda") for a in xi)
    deltas = [0.01 * torch.stack([a, -a]) for a in (xr, xa)]
    both = [a + d for a, d in zip((xr, xa), deltas)]
    graph = model.capture_grad()
    for other in (lambda: model.nll_and_grad(xr, xa), lambda: model.nll_and_grad_batch(*both),
                  graph.launch):
        other()
        with pytest.raises(RuntimeError, match="no sampled KL"):
            _kl_result(model, 2)
        nll, squares, _ = model.kl_and_grad(xr, xa, *deltas)
        assert _kl_result(model, 2) == (list(nll), squares)
