"""Chunk sizes of the surrogate's inference: any positive one gives the same rows, others are refused."""
import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("hidden", [(64, 64), (50,)])      # whole passes, layer by layer
def test_chunks(gpu, hidden):
    from holodeck_amd import surrogate as S
    net = S.MLPSurrogate(n_in=6, hidden=hidden, n_out=9, seed=2)
    net.x_lo, net.x_hi = np.zeros(6), np.ones(6)
    net.y_mean, net.y_std = np.zeros(9), np.ones(9)
    X = np.random.default_rng(0).random((37, 6))
    want = net.predict(X)
    for chunk in (1, 36, 37, 38):
        assert np.array_equal(net.predict(X, chunk=chunk), want)
    for chunk in (0, -1, -100):
        with pytest.raises(ValueError):
            net.predict(X, chunk=chunk)
