"""The training pass's loss (hd_mlp_train_step) against a 64-bit mean over the outputs it returns: rows off
the blocks of 16, outputs off the tiles of 16, one row, one output."""
import numpy as np
import pytest
import torch


def _net(n_in, hidden, n_out):
    from holodeck_amd import surrogate as S
    net = S.MLPSurrogate(n_in=n_in, hidden=hidden, n_out=n_out, seed=6)
    assert net._net() is not None
    return net


# FP32 rounding of one difference twice (squared) and its square, of at most 8 terms a lane, 6 levels of a
# wave, 8 waves, the scale, and one addition per block of 16 rows, all of one sign: (25 + rows / 16) 2^-24
@pytest.mark.gpu
@pytest.mark.parametrize("n_in,hidden,n_out,rows", [
    (6, (256, 256, 256, 256), 90, 1024), (6, (64, 64), 12, 17), (7, (32,), 1, 50), (6, (128, 96, 64), 256, 129),
    (3, (), 9, 64), (6, (32,) * 7, 33, 130), (6, (32,), 1, 1), (6, (64,), 17, 16), (6, (64,), 241, 15),
])
def test_loss_is_the_mean_square(gpu, n_in, hidden, n_out, rows):
    print(f"[mlp loss {n_in}-{hidden}-{n_out} rows={rows}]", flush=True)
    net = _net(n_in, hidden, n_out)
    rng = np.random.default_rng(rows)
    X, Y = rng.random((rows, n_in)).astype(np.float32), rng.normal(size=(rows, n_out)).astype(np.float32)
    loss, _, y = net.loss_and_grads(X, Y)
    want = np.mean((y.cpu().numpy().astype(float) - Y.astype(float)) ** 2)
    assert abs(float(loss) - want) <= (25 + rows / 16) * 2.0**-24 * want


@pytest.mark.gpu
@pytest.mark.parametrize("rows,batch", [(300, 129), (64, 512), (512, 128)])
def test_epoch_loss_counts_every_row_of_its_batches(gpu, rows, batch):
    """Without a step (lr = 0) the network stays, and the epoch's loss is the mean over the whole batches of
    the loss of their rows: over all rows where they fill the batches, else over those of the shuffle."""
    net = _net(6, (64, 64), 12)
    rng = np.random.default_rng(rows)
    X, Y = rng.random((rows, 6)), rng.normal(size=(rows, 12))
    hist = net.fit(X, Y, epochs=2, batch=batch, lr=0.0, seed=3)
    perms = []
    gen = torch.Generator(device="cpu").manual_seed(3)
    for _ in range(2):
        perms.append(torch.randperm(rows, generator=gen).numpy())
    x01 = torch.as_tensor(net._x01(X), dtype=torch.float32).cuda().to(torch.bfloat16)
    y = net.predict_device(x01.contiguous()).cpu().numpy().astype(float)
    t = ((Y - net.y_mean) / net.y_std).astype(np.float32).astype(float)
    for p, h in zip(perms, hist):
        whole = [p[s:s + batch] for s in range(0, rows - batch + 1 if rows >= batch else 1, batch)]
        want = np.mean([np.mean((y[i] - t[i]) ** 2) for i in whole])
        # as above, and the targets' own FP32 rounding (their mean and deviation are made on the device):
        # 2^-23 of targets of a few units in differences of about their size
        assert abs(h - want) <= ((25 + batch / 16) * 2.0**-24 + 2.0**-21) * want
