"""Drawn realizations where the work is cut: tiles per item, groups of the table-less records, long
tables built in parts.  The counts drawn are recorded; walking them as given counts gives the
outputs, and each bin's counts have its mean."""
import numpy as np
import pytest
import torch


# sizes: one tile and a bit; one bin; several tiles per item (enough items); realizations that leave
# one wave group, several, or a ragged last one; more than a workgroup has threads.  The tables of
# the widest kept window, the first bins without a table, and Normal draws are all among the means.
@pytest.mark.gpu
@pytest.mark.parametrize("B,F,R,L,mode,npar", [
    (700, 3, 64, 3, 0, 0), (1, 1, 1, 1, 0, 0), (513, 2, 257, 5, 1, 0), (512, 5, 100, 10, 0, 7), (1100, 1, 600, 16, 0, 0),
    (2600, 4, 129, 2, 1, 3), (900, 2, 65, 5, 2, 0), (700, 1, 200, 16, 1, 7), (530000, 12, 2, 1, 0, 0),
])
def test_drawn_counts_give_the_outputs(gpu, B, F, R, L, mode, npar):
    from holodeck_amd import _lib, engine
    from holodeck_amd import device as D
    print(f"[drawn items B={B} F={F} R={R} L={L} mode={mode} npar={npar}]", flush=True)
    rng = np.random.default_rng(B + F + R)
    lam = 10.0 ** rng.uniform(-2, 11, size=(B, F))
    lam[rng.random((B, F)) < 0.2] = 0.0
    lam.flat[:6] = [4.09e5, 4.1e5, 1e10, 1.01e10, 9.0, 2e9][:min(6, lam.size)]
    h = 10.0 ** rng.uniform(-12, -9, size=(B, F)) / (1.0 + lam)
    par = D.to_dev(rng.uniform(1.0, 2.0, size=(npar, B, F))) if npar else None
    n_d, h_d = D.to_dev(lam), D.to_dev(h)
    order = engine.order_desc(h_d, col=0) if mode == _lib.HD_SEL_SORTED else None
    rec = torch.empty((B, F, R), dtype=torch.float64, device="cuda")
    got = engine.realize(n_d, h_d, R, L, mode, order=order, par=par, seed=11, record_counts=rec)
    again = engine.realize(n_d, h_d, R, L, mode, order=order, par=par, seed=11)
    want = engine.realize(n_d, h_d, R, L, mode, order=order, par=par, counts=rec)
    for a, b in zip(got, again):
        assert a is None or torch.equal(a, b)
    # non-negative terms: any order of at most 530,000 of them agrees to 6e-11 of the total
    total = torch.einsum('bfr,bf->fr', rec, h_d)
    assert bool(((got[2] - want[2]).abs() <= 6e-11 * total).all())
    if mode != _lib.HD_SEL_NONE:
        assert torch.equal(got[1], want[1]) and torch.equal(got[0], want[0])
    if npar:
        some = want[2] > 1e-3 * total
        err = (got[3] - want[3]).abs()[:, some]
        assert bool((err <= 1e-6 * want[3].abs()[:, some]).all())
    if B <= 3000:
        # 6 standard errors of a mean of R draws (one in 1e9 bins), widened for the skewed small means
        dev = (rec.mean(dim=2) - n_d).abs()
        assert bool((dev <= 6.0 * torch.sqrt(n_d / R) + 12.0 / R).all())
        assert bool((rec[n_d == 0] == 0).all())


# counts summed of 257 (the first wave build), just below and above the split (2048) and the widest
@pytest.mark.gpu
@pytest.mark.parametrize("lam", [400.0, 430.0, 2.44e4, 2.46e4, 2.5e4, 9.9e4, 4.05e5])
def test_long_tables_match_the_poisson_cdf(gpu, lam):
    from scipy.stats import poisson
    from holodeck_amd import _lib
    from holodeck_amd import device as D
    cap = 6392
    kn = torch.zeros(3, dtype=torch.int32, device="cuda")
    cdf = torch.zeros(cap, dtype=torch.int64, device="cuda")
    _lib.call("hd_poisson_cdf_table", float(lam), cap, D.ptr(kn), D.ptr(cdf), D.stream_ptr())
    kb, kt, n = (int(v) for v in kn.cpu())
    F = cdf[:n].cpu().numpy().view(np.uint64)
    print(f"[long table lam={lam}: {kt + n - kb} counts]", flush=True)
    assert np.all(F[1:] >= F[:-1])
    want = poisson.cdf(kt + np.arange(n), lam) - poisson.cdf(kb - 1, lam)
    # a sum of positive terms: about one ulp per count, then rounded down to a multiple of 2^-64
    # (scipy's own incomplete gamma is good to about 1e-12 at these means)
    assert np.all(np.abs(F / 2.0**64 - want) <= 1e-11 * want + 2.0**-63)
