"""The pipelined Gauss-Seidel sweeps against the sequential ones (both reproduce scipy's update order, so
the gradients and sweep counts are equal to the last bit) over grids whose steps, rings and workgroups
differ: few vertices, steps of more than 128 vertices, long and short periods."""
import numpy as np
import pytest

from holodeck_amd.constants import MSOL


@pytest.mark.gpu
@pytest.mark.parametrize("M,Q", [(2, 2), (2, 9), (9, 2), (5, 4), (17, 15), (150, 30), (200, 30), (30, 90), (41, 81), (91, 81)])
def test_pipelined_sweeps_equal_sequential_ones(gpu, M, Q):
    from holodeck_amd import device as D, scatter
    rng = np.random.default_rng(M * 100 + Q)
    mtot, mrat = np.logspace(4, 12, M) * MSOL, np.logspace(-3, 0, Q)
    lm = np.log10(mtot / MSOL)[:, None, None]
    dens = np.repeat(10 ** (-0.4 * (lm - 8)) * np.exp(-10 ** (lm - 9)) * (1 + mrat[None, :, None]), 6, axis=2)
    dens *= 10 ** rng.uniform(-3, 3, size=6)
    dens *= 1 + 0.3 * rng.standard_normal(dens.shape)
    dens[:, :, 1] = 0.0                                  # nothing to do
    dens[:, :, 2] = 3.0                                  # all differences zero
    dens[: M // 2, :, 3] = 0.0                           # exact zeros beside numbers
    dens[:, :, 4] *= 1e-300
    dens[:, :, 5] *= 1e280
    keep = scatter.PIPELINED_SWEEPS
    try:
        for maxiter in (1, 2, 400):
            print(f"[ct pipe {M}x{Q} maxiter={maxiter}]", flush=True)
            got = []
            for pipelined in (True, False):
                scatter.PIPELINED_SWEEPS = pipelined
                it, gr = scatter.add_scatter_to_masses_device(mtot, mrat, D.to_dev(dens), 0.3, maxiter=maxiter,
                                                              return_grads=True)
                got.append((D.to_host(it)[:-1], D.to_host(gr).view(np.int64)))
            assert np.array_equal(got[0][0], got[1][0])
            assert np.array_equal(got[0][1], got[1][1])
    finally:
        scatter.PIPELINED_SWEEPS = keep
