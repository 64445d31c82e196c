"""Integration and strain where their threads' redshift groups end: a grid's result equals that of its
redshift bins taken one at a time (to the last bit: the operations of an output are the same), and the
integration a numpy sum over the corners (eight non-negative terms and four factors: within 16 ulp)."""
import numpy as np
import pytest

from holodeck_amd.constants import MSOL


@pytest.mark.gpu
@pytest.mark.parametrize("M,Q,Z,F", [(2, 2, 2, 1), (3, 2, 3, 5), (2, 4, 4, 257), (5, 3, 5, 40), (3, 3, 6, 64), (4, 2, 9, 1),
                                     (3, 4, 10, 300), (2, 3, 101, 7)])
def test_groups_of_redshift_bins(gpu, M, Q, Z, F):
    import holodeck_amd as holo
    from holodeck_amd import device as D, engine
    print(f"[bin items M={M} Q={Q} Z={Z} F={F}]", flush=True)
    rng = np.random.default_rng(Z * 1000 + F)
    cos = holo.Cosmology()
    lm, mr = np.linspace(37.0, 45.0, M), np.logspace(-2, 0, Q)
    rz, dl = np.logspace(-2, 1, Z), rng.uniform(0.01, 0.1, size=F)
    dn = 10.0 ** rng.uniform(-20, 20, size=(M, Q, Z, F))
    rf = rng.uniform(0.0, 5.0, size=(M, Q, Z, F))
    rf[rng.random(rf.shape) < 0.3] = -1.0
    fc = np.logspace(-9, -7, F)
    mc, qc = np.logspace(6, 10, M - 1) * MSOL, np.logspace(-2, 0, Q - 1)
    both = []
    for cut in ([(0, Z)], [(z, z + 2) for z in range(Z - 1)]):
        num = [D.to_host(engine.integrate_3dx1d(D.to_dev(lm), D.to_dev(mr), D.to_dev(rz[a:b]), D.to_dev(dl),
                                                D.to_dev(dn[:, :, a:b].copy()))) for a, b in cut]
        h2 = [D.to_host(engine.h2fdf_redz(D.to_dev(mc), D.to_dev(qc), D.to_dev(fc), D.to_dev(fc / 1e-9),
                                          D.to_dev(rf[:, :, a:b].copy()), cos)) for a, b in cut]
        both.append((np.concatenate(num, axis=2), np.concatenate(h2, axis=2)))
    assert np.array_equal(both[0][0], both[1][0])
    assert np.array_equal(both[0][1], both[1][1])
    want = sum(dn[i:M - 1 + i, j:Q - 1 + j, k:Z - 1 + k] for i in (0, 1) for j in (0, 1) for k in (0, 1)) / 8.0
    want = want * np.diff(lm)[:, None, None, None] * np.diff(mr)[:, None, None] * np.diff(rz)[:, None] * dl
    assert np.allclose(both[0][0], want, rtol=16 * 2.0**-52, atol=0)
