"""hd_gemm_f64 over its two kernels and their edges, against numpy: each output within twice the bound
(k + 1) 2^-53 sum |a b| of a sum of k products in any order."""
import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (65, 63, 17), (1023, 1024, 5), (1024, 1024, 16), (1025, 1025, 15), (129, 8200, 33),
                                   (364, 5001, 364), (8191, 129, 1), (127, 8300, 100), (2, 530000, 3)])
def test_gemm_f64(gpu, m, n, k):
    import torch
    from holodeck_amd import _lib
    from holodeck_amd import device as D
    print(f"[gemm {m}x{n}x{k}]", flush=True)
    rng = np.random.default_rng(m + n + k)
    a = rng.standard_normal((m, k)) * 10.0 ** rng.uniform(-3, 3, size=(m, 1))
    b = rng.standard_normal((k, n)) * 10.0 ** rng.uniform(-3, 3, size=(k, 1))
    c = torch.full((m, n), float("nan"), dtype=torch.float64, device="cuda")
    a_d, b_d = D.to_dev(a), D.to_dev(b)
    _lib.call("hd_gemm_f64", D.ptr(a_d), D.ptr(b_d), D.ptr(c), m, n, k, D.stream_ptr())
    assert np.all(np.abs(D.to_host(c) - a @ b) <= 2 * (k + 1) * 2.0**-53 * (np.abs(a) @ np.abs(b)))
