"""The read-out by a list of kept positions (jubik_readout_gather and its
transpose, called through the C ABI only) against boolean indexing and against
the read-out by bit words."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pixels", [1, 255, 257, 4099])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("keep", [0.0, 0.5, 1.0])
def test_list_equals_words(ja, pixels, dtype, keep):
    rng = np.random.default_rng(pixels)
    kept = rng.random(pixels) < keep
    x = torch.as_tensor(rng.standard_normal(pixels), dtype=dtype, device="cuda")
    index = torch.as_tensor(np.flatnonzero(kept), device="cuda")
    code, p = int(dtype == torch.float64), lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
    out = torch.empty(index.numel(), dtype=dtype, device="cuda")
    ja._lib.call("jubik_readout_gather", code, p(x), p(index), index.numel(), p(out), None)
    back = torch.empty_like(x)
    ja._lib.call("jubik_readout_scatter", code, p(out), p(index), index.numel(), pixels, p(back),
                 None)
    torch.cuda.synchronize()
    on = torch.as_tensor(kept, device="cuda")
    assert torch.equal(out, x[on])
    assert torch.equal(back, torch.where(on, x, torch.zeros_like(x)))
    ro = ja.build_readout_function(kept.astype(float).reshape(1, 1, 1, -1), keys=["a"])
    vec = ro(x.reshape(1, 1, 1, -1))
    assert torch.equal(vec["a"], out)
    assert torch.equal(ro.transpose(vec).reshape(-1), back)
