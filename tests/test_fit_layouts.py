"""Training takes its arrays in any layout: rows, columns (Fortran order), strided views, lists, FP32."""
import numpy as np
import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("hidden", [(64, 32), (50,)])      # whole passes, layer by layer
@pytest.mark.parametrize("batch", [16, 64])                # several batches; one, with all rows
def test_layouts_train_alike(gpu, hidden, batch):
    from holodeck_amd import surrogate as S
    rng = np.random.default_rng(8)
    X = rng.random((40, 6)).astype(np.float32).astype(float)
    Y = rng.normal(size=(40, 5)).astype(np.float32).astype(float)
    wide = np.zeros((80, 12))
    wide[::2, ::2] = X

    def train(x, y):
        net = S.MLPSurrogate(n_in=6, hidden=hidden, n_out=5, seed=3)
        net.fit(x, y, epochs=2, batch=batch, lr=1e-2, seed=1)
        return [t.cpu() for t in (*net.W, *net.b)] + [torch.as_tensor(net.predict(x))]

    want = train(X, Y)
    for x, y in ((np.asfortranarray(X), Y), (X, np.asfortranarray(Y)), (np.asfortranarray(X), np.asfortranarray(Y)),
                 (wide[::2, ::2], Y), (X[::-1][::-1], Y), (X.tolist(), Y.tolist()),
                 (X.astype(np.float32), Y.astype(np.float32))):
        for got, ref in zip(train(x, y), want):
            assert torch.equal(got, ref)


@pytest.mark.gpu
def test_gradients_of_any_layout(gpu):
    from holodeck_amd import surrogate as S
    rng = np.random.default_rng(9)
    X, Y = rng.random((33, 6)), rng.normal(size=(33, 5))
    net = S.MLPSurrogate(n_in=6, hidden=(64,), n_out=5, seed=3)
    _, ref, y_ref = net.loss_and_grads(X, Y)
    for x, y in ((np.asfortranarray(X), np.asfortranarray(Y)), (torch.as_tensor(X).t().contiguous().t(), torch.as_tensor(Y))):
        _, got, out = net.loss_and_grads(x, y)
        assert torch.equal(out, y_ref)
        for (dW, db), (rW, rb) in zip(got, ref):
            assert torch.equal(dW, rW) and torch.equal(db, rb)
