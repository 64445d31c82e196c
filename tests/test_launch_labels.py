"""Launch timing tells a network's whole pass from its layers' products."""
import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("hidden,label,other,launches", [((64, 64), "k_mlp_forward", "k_mlp_gemm", 1),
                                                         ((50, 50), "k_mlp_gemm", "k_mlp_forward", 3)])
def test_inference_is_timed_under_its_kernel(gpu, hidden, label, other, launches):
    from holodeck_amd import _lib, surrogate
    net = surrogate.MLPSurrogate(n_in=6, hidden=hidden, n_out=9, seed=2)
    X = np.random.default_rng(0).random((20, 6))
    _lib.timing_enable(True)
    try:
        net.predict(X)
        ms, n = _lib.timing_read(label)
        assert n == launches and ms > 0.0 and _lib.timing_read(other) == (0.0, 0)
    finally:
        _lib.timing_enable(False)
