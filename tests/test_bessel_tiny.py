"""The Bessel pair at high orders and tiny arguments, where a term of the backward recurrence is up to 2e17
times the one before it: the values underflow, to zero and not to NaN."""
import numpy as np
import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("lo", [100, 248, 249, 5000, 58000, 60000, 70000, 99999, 100000])
def test_underflow_is_zero(gpu, lo):
    from holodeck_amd import _lib
    from holodeck_amd import device as D
    line = 4e-15 * (max(lo, 249) + 2)     # below it the recurrence looks for overflow at every step
    x = np.concatenate([[1e-12, 1.0000001e-12, 1.5e-12, 0.999999999 * line, line, 1.000000001 * line],
                        10.0 ** np.linspace(-12, -6, 61)])
    print(f"[bessel pair lo={lo}, {x.size} tiny arguments]", flush=True)
    lo_d = torch.full((x.size,), lo, dtype=torch.int32, device="cuda")
    x_d, out = D.to_dev(x), D.empty((x.size, 2))
    _lib.call("hd_bessel_jpair", D.ptr(lo_d), D.ptr(x_d), x.size, D.ptr(out), D.stream_ptr())
    assert np.all(D.to_host(out) == 0.0)
