"""Eccentric sums where the kernels divide their work: the Bessel pair's two start rules, evolutions
longer than the LDS copy, mass-ratio grids longer than one LDS batch, ragged redshift groups."""
import numpy as np
import pytest
import torch


# orders around the change of the start rule (6), arguments below, at and beyond the turning point, and
# the tiny ones that grow fastest.  A backward recurrence is exact to a few ulp per step of the larger
# of the pair: (order + 100) 2^-51; underflowing values aside.  scipy's jv, good to 1e-12 in the tests of
# this range but not to that beyond the turning point, is asked first and mpmath where it disagrees.
@pytest.mark.gpu
@pytest.mark.parametrize("lo", [-1, 0, 3, 5, 6, 7, 8, 9, 10, 16, 17, 60, 98, 500])
def test_bessel_pair_at_the_start_rules(gpu, lo):
    from scipy.special import jv
    from holodeck_amd import _lib
    from holodeck_amd import device as D
    rng = np.random.default_rng(lo + 2)
    x = np.concatenate([(lo + 2) * 10.0 ** rng.uniform(-13, 0, 200), (lo + 2) * rng.uniform(0.1, 1.0, 300),
                        (lo + 2) * rng.uniform(1.0, 5.0, 100)])
    print(f"[bessel pair lo={lo}]", flush=True)
    lo_d = torch.full((x.size,), lo, dtype=torch.int32, device="cuda")
    x_d, out = D.to_dev(x), D.empty((x.size, 2))
    _lib.call("hd_bessel_jpair", D.ptr(lo_d), D.ptr(x_d), x.size, D.ptr(out), D.stream_ptr())
    got, want = D.to_host(out), np.stack([jv(lo, x), jv(lo + 1, x)], axis=1)
    scale = np.abs(want).max(axis=1)
    ok = scale > 1e-280
    err = np.abs(got - want).max(axis=1)
    tol = 1e-12 + (abs(lo) + 100) * 2.0**-51
    import mpmath
    with mpmath.workdps(30):
        for i in np.flatnonzero(ok & ~(err <= tol * scale)):
            want[i] = [float(mpmath.besselj(lo + d, mpmath.mpf(x[i]))) for d in (0, 1)]
    err = np.abs(got - want).max(axis=1)
    assert np.all(err[ok] <= tol * scale[ok]), (err[ok] / scale[ok]).max()


@pytest.mark.gpu
@pytest.mark.parametrize("M,Q,Z,F,H,E", [(3, 2, 2, 1, 3, 2), (5, 257, 65, 2, 20, 100), (4, 300, 130, 3, 4, 2049), (2, 9, 64, 2, 5, 2048)])
def test_sums_match_the_nodes(gpu, M, Q, Z, F, H, E):
    """The spectrum equals the sum over nodes of Poisson mean times strain factor (hd_eccen_number),
    which evaluates every node on its own: the terms are of one sign, so both sums are good to a few
    hundred ulp of their largest."""
    from holodeck_amd import cyutils, engine
    rng = np.random.default_rng(M + Q)
    ndens = 10.0 ** rng.uniform(-8, -3, size=(M, Q, Z))
    ndens[rng.random(ndens.shape) < 0.3] = 0.0
    lm = np.log10(2e33) + np.linspace(6, 10, M)
    mrat, redz = np.logspace(-2, 0, Q), np.logspace(-2, 0.8, Z)
    dcom = 4000.0 * np.log1p(redz)
    sepa = np.logspace(np.log10(3e18), 14, E)
    eccen = np.linspace(0.7, 0.2, E)
    fobs = np.array([2e-9, 1.1e-8, 4e-8])[:F]
    args = cyutils._eccen_dev(ndens, lm, mrat, redz, dcom, fobs, sepa, eccen)
    print(f"[eccentric sums {M}x{Q}x{Z} F={F} H={H} E={E}]", flush=True)
    got = engine.gwb_eccen(*args, H)
    lam, hval = engine.eccen_number(*args, 0, H)
    want = (lam * hval).sum(dim=0).view(F, H)
    assert bool((want > 0).any())
    assert bool(((got - want).abs() <= 1e-11 * want).all())
