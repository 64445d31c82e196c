"""Whole passes of the surrogate (hd_mlp_forward, hd_mlp_train_step) against the layer-by-layer kernels,
which test_surrogate.py holds to FP32 references: the same products summed in the same order, so the
outputs, the gradients and the updated weights are equal; the loss adds its terms in any order."""
import numpy as np
import pytest
import torch


def _pair(n_in, hidden, n_out, seed=4):
    from holodeck_amd import surrogate as S
    a = S.MLPSurrogate(n_in=n_in, hidden=hidden, n_out=n_out, seed=seed)
    b = S.MLPSurrogate(n_in=n_in, hidden=hidden, n_out=n_out, seed=seed)
    rng = np.random.default_rng(seed)
    for net in (a, b):
        for l, v in enumerate(net.b):
            v.copy_(torch.as_tensor(rng.normal(size=v.numel()).astype(np.float32) if net is a else a.b[l].cpu()))
        net.x_lo, net.x_hi = -np.arange(1.0, n_in + 1), np.arange(1.0, n_in + 1)
        net.y_mean, net.y_std = np.linspace(-15, -13, n_out), np.linspace(0.3, 0.9, n_out)
    assert a._net() is not None
    b._net = lambda: None
    return a, b, rng


# widths at both ends, inputs and outputs off the multiples of 16 and 32, one layer and eight, an output
# wider than one round of tiles; rows around a block (16), around the switch of block height (8192)
@pytest.mark.gpu
@pytest.mark.parametrize("n_in,hidden,n_out,rows", [
    (6, (256, 256, 256, 256), 90, 1), (7, (256,) * 4, 120, 17), (6, (32,), 1, 15), (1, (64, 96), 33, 16),
    (40, (128,) * 7, 16, 63), (6, (), 5, 100), (6, (256, 64), 300, 65), (6, (64, 256), 90, 8192),
    (6, (256, 256), 90, 8193), (13, (32, 32), 513, 8250),
])
def test_forward_equals_the_layers(gpu, n_in, hidden, n_out, rows):
    print(f"[mlp forward {n_in}-{hidden}-{n_out} rows={rows}]", flush=True)
    a, b, rng = _pair(n_in, hidden, n_out)
    x = torch.as_tensor(rng.random((rows, n_in)).astype(np.float32)).cuda().to(torch.bfloat16)
    assert torch.equal(a.predict_device(x), b.predict_device(x))
    X = a.x_lo + (a.x_hi - a.x_lo) * rng.random((rows, n_in))
    assert np.array_equal(a.predict(X), b.predict(X))
    assert np.array_equal(a.predict(X, chunk=max(rows // 3, 1)), b.predict(X))


@pytest.mark.gpu
@pytest.mark.parametrize("n_in,hidden,n_out,rows,batch", [
    (6, (256, 256, 256, 256), 90, 2048, 1024), (6, (64, 64), 12, 300, 512), (7, (32,), 1, 50, 17),
    (6, (128, 96, 64), 256, 700, 129), (3, (), 9, 64, 16), (6, (32,) * 7, 33, 130, 128),
])
def test_training_equals_the_layers(gpu, n_in, hidden, n_out, rows, batch):
    print(f"[mlp training {n_in}-{hidden}-{n_out} rows={rows} batch={batch}]", flush=True)
    a, b, rng = _pair(n_in, hidden, n_out)
    X, Y = rng.random((rows, n_in)), rng.normal(size=(rows, n_out))
    la, ga, ya = a.loss_and_grads(X[:batch], Y[:batch])
    lb, gb, yb = b.loss_and_grads(X[:batch], Y[:batch])
    assert torch.equal(ya, yb)
    # FP32 sums of at most 262,144 squares in different orders: n eps / 2 bounds the relative difference
    assert abs(float(la) - float(lb)) <= 0.02 * float(lb)
    for l, ((dW, db), (rW, rb)) in enumerate(zip(ga, gb)):
        assert torch.equal(dW, rW) and torch.equal(db, rb), l
    assert a.step == 0
    ha = a.fit(X, Y, epochs=2, batch=batch, lr=1e-3)
    hb = b.fit(X, Y, epochs=2, batch=batch, lr=1e-3)
    assert np.allclose(ha, hb, rtol=0.02)
    assert a.step == b.step
    for l in range(a.nlayers):
        for u, v in ((a.W, b.W), (a.b, b.b), (a.Wb, b.Wb), (a.mW, b.mW), (a.vW, b.vW), (a.mb, b.mb), (a.vb, b.vb)):
            assert torch.equal(u[l], v[l]), l


@pytest.mark.gpu
def test_networks_the_passes_do_not_take(gpu):
    """Hidden widths off 32 or above 256 and inputs above 256 run layer by layer; a network with more than
    256 outputs trains layer by layer."""
    from holodeck_amd import surrogate as S
    rng = np.random.default_rng(1)
    for n_in, hidden, n_out in ((6, (50,), 4), (6, (288,), 4), (300, (64,), 4)):
        net = S.MLPSurrogate(n_in=n_in, hidden=hidden, n_out=n_out)
        assert net._net() is None
        assert net.predict(rng.random((5, n_in))).shape == (5, n_out)
        net.fit(rng.random((40, n_in)), rng.random((40, n_out)), epochs=1, batch=16)
    net = S.MLPSurrogate(n_in=6, hidden=(64,), n_out=300)
    net.fit(rng.random((40, 6)), rng.random((40, 300)), epochs=1, batch=16)
    assert net.step == 2
