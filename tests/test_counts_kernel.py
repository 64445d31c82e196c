"""Realizations of given counts (hd_realize_counts) where the launch is cut: column blocks, bin
chunks, the merge's groups, list capacities, against a numpy walk over the same counts."""
import numpy as np
import pytest


def _walk(counts, h, order_of, L, skip_below):
    """First L instances per (f, r) in the order's priority; the rest of sum(n h) is background."""
    B, F, R = counts.shape
    ss = np.zeros((F, R, L))
    idx = np.full((F, R, L), -1, dtype=np.int64)
    n = np.where(counts < 1, 0.0, counts) if skip_below else counts
    bg = np.einsum('bfr,bf->fr', n, h)
    for f in range(F):
        order = order_of(f)
        for r in range(R):
            left = np.minimum(np.ceil(n[order, f, r]), L).astype(int)
            hit = np.flatnonzero(left > 0)[:L]
            bins = np.repeat(order[hit], left[hit])[:L]
            idx[f, r, :bins.size] = bins
            ss[f, r, :bins.size] = h[bins, f]
    return ss, idx, bg - ss.sum(axis=-1)


# tolerance: n h are non-negative, so a sum of B <= 5000 terms in any order is exact to B ulp
# (5000 * 2^-53 < 6e-13); the background subtracts the loud terms from it
@pytest.mark.gpu
@pytest.mark.parametrize("B,F,R,L,mode,npar", [
    (1, 1, 1, 1, 0, 0), (7, 3, 5, 3, 0, 0), (64, 2, 32, 5, 1, 0), (65, 5, 51, 10, 0, 0), (521, 1, 257, 1, 1, 0),
    (4999, 7, 9, 16, 0, 0), (4097, 3, 1, 5, 0, 7), (1200, 4, 65, 2, 1, 3), (3001, 9, 30, 5, 2, 0), (5000, 2, 3, 16, 1, 8),
])
def test_given_counts_match_a_numpy_walk(gpu, B, F, R, L, mode, npar):
    from holodeck_amd import _lib, engine
    from holodeck_amd import device as D
    print(f"[given counts B={B} F={F} R={R} L={L} mode={mode} npar={npar}]", flush=True)
    rng = np.random.default_rng(B + 31 * F + R)
    lam = 10.0 ** rng.uniform(-3, 1.5, size=(B, F))
    counts = rng.poisson(lam[..., None], size=(B, F, R)).astype(float)
    if mode == 0:                      # Normal draws of very large bins are not whole and may fall below one
        counts[::5] = np.maximum(counts[::5] + rng.uniform(-0.7, 0.7, size=counts[::5].shape), 0.0)
    h = 10.0 ** rng.uniform(-3, 0, size=(B, F))
    h[rng.random((B, F)) < 0.1] = 0.5  # equal strains: the lower bin first
    par = rng.uniform(1.0, 2.0, size=(npar, B, F)) if npar else None
    h_d, c_d = D.to_dev(h), D.to_dev(counts)
    order = np.argsort(-h[:, 0], kind='stable')
    ss, idx, bg, bgpar = engine.realize(None, h_d, R, L, mode, order=D.to_dev(order) if mode == _lib.HD_SEL_SORTED else None,
                                        counts=c_d, par=D.to_dev(par) if npar else None)
    total = np.einsum('bfr,bf->fr', np.where(counts < 1, 0.0, counts) if mode == 0 else counts, h)
    if mode == _lib.HD_SEL_NONE:
        assert np.allclose(D.to_host(bg), total, rtol=1e-12, atol=0)
        return
    order_of = (lambda f: order) if mode == _lib.HD_SEL_SORTED else (lambda f: np.argsort(-h[:, f], kind='stable'))
    w_ss, w_idx, w_bg = _walk(counts, h, order_of, L, mode == _lib.HD_SEL_SORTED)
    assert np.array_equal(D.to_host(idx), w_idx)
    assert np.array_equal(D.to_host(ss), w_ss)
    assert np.all(np.abs(D.to_host(bg) - w_bg) <= 1e-12 * total)
    if npar:
        n = np.where(counts < 1, 0.0, counts) if mode == 0 else counts
        for k in range(npar):
            sel = np.zeros((F, R))
            for j in range(L):
                ok = w_idx[..., j] >= 0
                sel += np.where(ok, w_ss[..., j] * par[k][np.where(ok, w_idx[..., j], 0), np.arange(F)[:, None]], 0.0)
            want = np.einsum('bfr,bf->fr', n, h * par[k]) - sel
            got = D.to_host(bgpar)[k]
            some = (w_idx[..., 0] >= 0) | (mode == _lib.HD_SEL_SORTED)
            some &= w_bg > 1e-9 * total
            assert np.all(np.abs(got * D.to_host(bg) - want)[some] <= 4e-12 * total[some])
