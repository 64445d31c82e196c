"""The step window of hd_dbn_2pwl: with sorted targets only the steps that can hold one are walked; a
call that does not promise sorted targets walks every step.  Both must record the same steps, so the
results are equal to the last bit."""
import numpy as np
import pytest

from holodeck_amd.constants import GYR, MSOL, PC, YR


@pytest.mark.gpu
@pytest.mark.parametrize("M,Q,Z,F,steps,sepa_pc,lo,hi", [
    (5, 4, 9, 6, 300, 1e4, -9.0, -7.5),       # the usual range
    (4, 3, 101, 40, 300, 1e4, -8.8, -7.1),
    (3, 2, 300, 5, 97, 1e3, -9.5, -6.0),      # more redshifts than threads: one share each
    (6, 3, 17, 1, 300, 1e4, -8.0, -8.0),      # one target
    (6, 3, 7, 9, 1, 1e4, -9.0, -7.0),         # one step
    (6, 3, 20, 8, 1200, 1e2, -13.0, -2.0),    # targets before the first step and past the last
    (6, 3, 20, 8, 64, 0.05, -9.0, -5.0),      # starts inside the ISCO of the heaviest: runs outwards
    (4, 3, 33, 1100, 50, 1e4, -9.0, -7.0),    # targets outside LDS
])
def test_sorted_targets_equal_the_walk_of_every_step(gpu, M, Q, Z, F, steps, sepa_pc, lo, hi):
    import holodeck_amd as holo
    from holodeck_amd import device as D, engine
    print(f"[dbn window M={M} Q={Q} Z={Z} F={F} steps={steps} sepa={sepa_pc}]", flush=True)
    rng = np.random.default_rng(steps + 7 * F + Z)
    cos = holo.Cosmology()
    mtot = np.logspace(5, 12, M) * MSOL
    mrat = np.logspace(-2, 0, Q)
    redz = np.logspace(-3, 1, Z)
    # lifetimes from far shorter to far longer than the age of the universe, no growth among them
    norm = 10.0 ** rng.uniform(-12, 12, size=M * Q)
    norm[0], norm[-1] = 0.0, 1e-20
    gmt = rng.uniform(0.0, 3.0, size=(M, Q, Z)) * GYR
    gmt[rng.random(gmt.shape) < 0.2] = 0.0
    gmt[rng.random(gmt.shape) < 0.1] = 20.0 * GYR
    fobs = np.logspace(lo, hi, F)
    if F > 3:
        fobs[2] = fobs[1]
    dens = rng.uniform(0.1, 1.0, size=(M, Q, Z))
    args = (float(sepa_pc * PC), steps, D.to_dev(norm), 100.0 * PC, -1.0, 1.5, D.to_dev(dens), D.to_dev(mtot),
            D.to_dev(mrat), D.to_dev(redz), D.to_dev(gmt), cos)
    got = [D.to_host(t) for t in engine.dbn_2pwl(D.to_dev(fobs), True, *args)]
    want = [D.to_host(t) for t in engine.dbn_2pwl(D.to_dev(fobs), False, *args)]
    assert np.array_equal(got[0], want[0], equal_nan=True)
    assert np.array_equal(got[1], want[1], equal_nan=True)
    if sepa_pc > 1 and hi < -6:
        assert np.any(want[0] > 0.0)
