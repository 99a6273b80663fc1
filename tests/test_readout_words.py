"""The bit words of the read-out against boolean indexing, on the host, with
no function of numpy newer than 1.22."""
import numpy as np
import pytest

import __graft_entry__


@pytest.mark.parametrize("shape", [(1, 1, 8, 8), (2, 3, 5, 7), (7, 1, 9, 64), (3, 2, 0, 4)])
@pytest.mark.parametrize("keep", [0.0, 0.5, 1.0])
def test_kept_words(monkeypatch, shape, keep):
    monkeypatch.delattr(np, "bitwise_count", raising=False)
    ja = __graft_entry__.load_package()
    rng = np.random.default_rng(3)
    kept = rng.random(shape) < keep
    words, counts = ja.response.kept_words(kept)
    per = int(np.prod(shape[1:]))
    assert words.shape == (2, shape[0], (per + 63) // 64) and words.dtype == np.int64
    for i in range(shape[0]):
        flat = kept[i].reshape(-1)
        assert counts[i] == flat.sum()
        bits = np.array([(int(w) >> b) & 1 for w in words[0, i] for b in range(64)], dtype=bool)
        np.testing.assert_array_equal(bits[:per], flat)
        assert not bits[per:].any()
        before = [flat[:64 * k].sum() for k in range(words.shape[2])]
        np.testing.assert_array_equal(words[1, i], before)
