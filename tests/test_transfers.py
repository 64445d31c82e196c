"""Host <-> device copies through the pinned slots, around the sizes where they are cut."""
import threading

import numpy as np
import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("nbytes", [8, (64 << 10) - 8, 64 << 10, (256 << 10) + 8, (4 << 20) - 8, 4 << 20, (4 << 20) + 8,
                                    (12 << 20) + 40])
def test_round_trip(gpu, nbytes):
    from holodeck_amd import device as D
    a = np.random.default_rng(nbytes).normal(size=nbytes // 8)
    t = D.to_dev(a)
    assert t.shape == a.shape and t.dtype == torch.float64
    assert np.array_equal(D.to_host(t), a)
    assert np.array_equal(D.to_host(t * 2.0 / 2.0), a)              # after work still queued on the stream
    assert np.array_equal(D.to_host(t.view(-1, 1).expand(-1, 2)), np.stack([a, a], axis=1))
    out = np.zeros((3, a.size))
    assert D.to_host(t, out=out[1]).base is not None and np.array_equal(out[1], a) and not out[[0, 2]].any()
    i = np.arange(nbytes // 8)
    assert np.array_equal(D.to_host(D.to_dev(i)), i)


@pytest.mark.gpu
def test_threads_on_their_own_streams(gpu):
    """Several threads at once: one holds the slots, the others take the runtime's copies."""
    from holodeck_amd import device as D
    bad = []

    def work(seed):
        rng = np.random.default_rng(seed)
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(8):
                a = rng.normal(size=1 << 20)
                if not np.array_equal(D.to_host(D.to_dev(a) + 1.0), a + 1.0):
                    bad.append(seed)

    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


@pytest.mark.gpu
@pytest.mark.parametrize("nbytes", [8, (256 << 10) + 8, (4 << 20) - 8, 4 << 20, (12 << 20) + 40])
def test_uploads_through_the_slots(gpu, nbytes, monkeypatch):
    """Only a caller that asks for the slots takes them: their upload waits for the stream's earlier
    kernels, which callers with several streams in flight must not."""
    from holodeck_amd import device as D
    a = np.random.default_rng(nbytes).normal(size=nbytes // 8)
    taken = []
    push = D._SLOTS.push
    monkeypatch.setattr(D._SLOTS, "push", lambda *args: taken.append(1) or push(*args))
    assert np.array_equal(D.to_host(D.to_dev(a)), a) and not taken
    assert np.array_equal(D.to_host(D.to_dev(a, slots=True)), a)
    assert len(taken) == (1 if nbytes > D.STAGE_MAX_BYTES else 0)
