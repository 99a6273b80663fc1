"""Read-out and Poisson energy of all modules in one launch: the kept pixels by
bit words against numpy's boolean indexing, the energies against the call for
one array; both copy and sum in a fixed order, so the comparisons are exact."""
import ctypes as C

import numpy as np
import pytest
import torch



def test_argument_checks(ja):
    lib = ja._lib.load()
    null, one = C.c_void_p(0), (C.c_void_p * 1)(8)
    gather, scatter = lib.jubik_readout_gather_words, lib.jubik_readout_scatter_words
    assert gather(2, 1, null, null, 1, null, 1, one, null) == ja._lib.EINVAL  # dtype
    assert gather(1, -1, null, null, 1, null, 1, one, null) == ja._lib.EINVAL
    assert gather(1, 1, null, null, 64, null, 63, one, null) == ja._lib.EINVAL  # x too short
    assert gather(1, 1, null, null, 64, null, 64, one, null) == ja._lib.EINVAL  # NULL
    assert scatter(1, 1, null, null, 64, one, null, null) == ja._lib.EINVAL
    nll = lib.jubik_poisson_nll_grad_segments
    n = (C.c_int64 * 1)(-1)
    assert nll(1, 1, one, one, n, C.c_void_p(8), None, C.c_void_p(8), null) == ja._lib.EINVAL
    assert nll(1, 1, None, one, n, C.c_void_p(8), None, C.c_void_p(8), null) == ja._lib.EINVAL


# pixels around one word, one wave's and one work-group's words; 16 modules
# fill a launch
@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1, 1, 1, 1), (2, 1, 7, 9), (1, 1, 8, 8), (1, 1, 5, 13),
                                   (3, 2, 16, 16), (2, 1, 19, 27), (2, 1, 32, 64), (1, 3, 23, 31),
                                   (16, 1, 6, 11), (17, 1, 6, 11), (33, 1, 3, 5)])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("keep", [0.0, 0.5, 1.0])
def test_readout_matches_boolean_indexing(ja, shape, dtype, keep):
    rng = np.random.default_rng(sum(shape))
    kept = rng.random(shape) < keep
    x = rng.standard_normal(shape).astype(dtype)
    keys = ["k%d" % i for i in range(shape[0])]
    ro = ja.build_readout_function(kept.astype(float), keys=keys)
    vec = ro(torch.as_tensor(x, device="cuda"))
    for i, k in enumerate(keys):
        np.testing.assert_array_equal(vec[k].cpu().numpy(), x[i][kept[i]])
    back = ro.transpose(vec)
    assert back.shape == shape and back.dtype == torch.as_tensor(x).dtype
    np.testing.assert_array_equal(back.cpu().numpy(), np.where(kept, x, 0))


@pytest.mark.gpu
def test_readout_of_some_modules_and_of_wrong_shapes(ja):
    flags = np.ones((3, 1, 4, 5))
    flags[0, 0, 1, 2] = 0
    ro = ja.build_readout_function(flags)  # no keys: the first module
    x = np.arange(60.0).reshape(3, 1, 4, 5)
    vec = ro(x)
    np.testing.assert_array_equal(vec["masked input"], np.delete(np.arange(20.0), 7))
    back = ro.transpose(vec)
    assert not back[1:].any()
    np.testing.assert_array_equal(back[0], np.where(flags[0] > 0, x[0], 0))
    ro = ja.build_readout_function(flags, keys=["a", "b", "c"])
    with pytest.raises(IndexError):
        ro(x[:2])
    with pytest.raises(ValueError):
        ro(x[:, :, :3])
    with pytest.raises(ValueError):
        ro.transpose({"a": np.ones(19), "b": np.ones(20), "c": np.ones(3)})


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [[1], [0, 5], [255, 256, 257], [300000, 1, 262144],
                                   list(range(1, 35))])
def test_energy_of_many_keys_is_the_sum_of_each(ja, sizes):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(len(sizes))
    lam, data = {}, {}
    for i, n in enumerate(sizes):  # every third key in the other element type
        dt = torch.float32 if i % 3 == 1 else torch.float64
        lam["k%d" % i] = torch.rand(n, generator=gen, device="cuda", dtype=dt) * 9 + 0.1
        data["k%d" % i] = torch.poisson(lam["k%d" % i], generator=gen)
    energy, grad = ja.Poissonian(ja.Vector(data)).energy_and_gradient(ja.Vector(lam))
    want = 0.0
    for k in lam:
        e, g = ja.Poissonian(data[k]).energy_and_gradient(lam[k])
        want += e
        assert grad[k].dtype == lam[k].dtype and torch.equal(grad[k], g)
        nll = torch.empty(1, dtype=torch.float64, device="cuda")
        work = torch.empty(ja._lib.POISSON_WORK_BYTES // 8, dtype=torch.float64, device="cuda")
        ja._lib.call("jubik_poisson_nll_grad", int(lam[k].dtype == torch.float64),
                     C.c_void_p(lam[k].data_ptr()), C.c_void_p(data[k].data_ptr()),
                     lam[k].numel(), C.c_void_p(nll.data_ptr()), None,
                     C.c_void_p(work.data_ptr()), None)
        torch.cuda.synchronize()
        assert float(nll) == e
    assert energy == want
