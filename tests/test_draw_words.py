"""The draw kernel's records in fours: the counts of every realization of a tile, recorded, against an
inversion of the same generator words on the host, record by record.  A wave in which one realization's
uniform falls outside a table redraws the pair exactly; the other realizations' counts, and
that one's after it, come from the words in the documented order (x_a, x_b, then w_a, w_b)."""
import numpy as np
import pytest
import torch


def _words(seed, tile, f, r, n):
    from holodeck_amd import _lib
    state = _lib.philox4x32_10([tile, f, r, 6 << 16], [seed & 0xffffffff, seed >> 32])
    if not any(state):
        state = [1, 0, 0, 0]
    return _lib.xoshiro128ss([int(v) for v in state], n)[1]


# one record to a whole batch of 128, over group remainders; few realizations, a full and a ragged wave
@pytest.mark.gpu
@pytest.mark.parametrize("B,R", [(1, 5), (2, 64), (3, 7), (4, 64), (5, 65), (6, 3), (7, 64), (8, 9), (9, 100), (128, 500), (127, 64)])
def test_counts_follow_the_words_in_order(gpu, B, R):
    from holodeck_amd import _lib, engine
    from holodeck_amd import device as D
    print(f"[draw words B={B} R={R}]", flush=True)
    rng = np.random.default_rng(B)
    lam = 10.0 ** rng.uniform(-0.2, 1.3, size=B)       # dense, and all tables of the tile in one batch
    seed = 0x123456789 + B
    rec = torch.empty((B, 1, R), dtype=torch.float64, device="cuda")
    h = D.to_dev(np.full((B, 1), 1e-30))
    engine.realize(D.to_dev(lam[:, None]), h, R, 1, _lib.HD_SEL_NONE, seed=seed, record_counts=rec)
    got = D.to_host(rec)[:, 0, :]
    tabs, total = [], 0
    for v in lam:
        kn = torch.zeros(3, dtype=torch.int32, device="cuda")
        cdf = torch.zeros(5120, dtype=torch.int64, device="cuda")
        _lib.call("hd_poisson_cdf_table", float(v), 5120, D.ptr(kn), D.ptr(cdf), D.stream_ptr())
        kb, kt, n = (int(x) for x in kn.cpu())
        tabs.append((kb, kt, n, [int(x) >> 32 for x in cdf[:n].cpu().numpy().view(np.uint64)]))
        total += n
    assert total <= 5120
    outside = 0
    for r in range(R):
        w = [int(x) for x in _words(seed, 0, 0, r, 2 * B + 2)]
        at = 0
        for a in range(0, B, 2):
            pair = range(a, min(a + 2, B))
            xs = w[at:at + len(pair)]
            at += len(pair)
            for i, x in zip(pair, xs):
                kb, kt, n, hi = tabs[i]
                j = int(np.searchsorted(hi, x, side='left'))     # first entry with high word >= x
                assert j >= n or hi[j] != x                      # (a tie: 2^-32, none for these seeds)
                if (j == 0 and kt > kb) or j == n:
                    outside += 1
                    at += 1                                      # the tail walk takes a second word
                    assert got[i, r] <= kt if j == 0 else got[i, r] >= kt + n - 1
                else:
                    assert got[i, r] == kt + j, (i, r)
    if B * R >= 30000:
        assert outside > 0
