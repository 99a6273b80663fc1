"""The inverse-gamma transform where its search changes method: the float
start ends at |xi| = 6 and at shape a = 64, the power series hands over to
the continued fraction at y = a + 1, and the table of reciprocals ends after
96 terms (a = 200).  Held to scipy's inverse incomplete gamma functions with
the tolerances of the transform's other tests."""
import numpy as np
import pytest
import torch

from oracle import points as op

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("a", [0.1, 0.999, 1.0, 1.995, 63.9, 64.1, 200.0])
@pytest.mark.parametrize("dtype,tol", [(torch.float64, 1e-12), (torch.float32, 2e-6)])
def test_search_switches(ja, a, dtype, tol):
    near6 = 6.0 + np.array([-1e-3, -1e-7, 0.0, 1e-7, 1e-3])
    xi = np.concatenate([near6, -near6, np.linspace(-7.0, 7.0, 141), [0.0, 1e-12, -1e-12]])
    prior = ja.priors.invgamma_prior(a, 1.0)
    x = torch.as_tensor(xi, dtype=dtype, device="cuda")
    logi, dlog = (v.double().cpu().numpy() for v in prior.log_and_dlog(x))
    xi = x.double().cpu().numpy()
    want = -np.log(op.invgamma_y(xi, a))
    assert np.max(np.abs(logi - want) / np.maximum(1.0, np.abs(want))) <= tol
    np.testing.assert_allclose(dlog, op.dlog_invgamma(xi, a, 1.0), rtol=max(tol, 1e-11) * 10)
