"""Many drawn realizations: what smaller items than 8 tiles add to the workspace stays bounded, and the
workgroups that share an item's realizations draw and sum each of them once."""
import numpy as np
import pytest
import torch


def _eight_tiles(B, F, R, L, npar):
    """Workspace with items of 8 tiles of 512 bins."""
    def up(n):
        return (n + 255) & ~255
    tiles = -(-B // 512)
    items = F * -(-tiles // 8)
    slots, parts, groups = 512 * F * tiles, items * R, 8 * F * R
    return (up(4 * B) + up(48 * 513 * F * tiles) + up(4 * 513 * F * tiles) + up(12 * F * tiles) + 3 * up(8 * slots) +
            2 * up(8 * slots * npar) + up(8 * parts) + up(8 * parts * npar) + up(8 * parts * L) + up(4 * parts * L) +
            up(groups * (8 + 8 * npar + 12 * L) + 1024) + 2 * up(4 * items) + up(4 * F * tiles) + 512)


@pytest.mark.parametrize("B", [1, 512, 2688, 120000, 720000, 5000000])
@pytest.mark.parametrize("F", [1, 6, 20, 40, 600])
@pytest.mark.parametrize("L,npar", [(0, 0), (5, 0), (10, 0), (16, 7)])
def test_workspace_stays_near_that_of_the_largest_items(B, F, L, npar):
    from holodeck_amd import _lib
    for R in (1, 100, 500, 513, 2000, 10000, 100000, 1000000):
        ws, eight = _lib.size("hd_realize_workspace_size", B, F, R, L, npar), _eight_tiles(B, F, R, L, npar)
        # fewer than 2 x 4096 x 512 partials of at most 256 bytes; up to 24 more groups to merge them, of
        # fewer than 8192 columns; the plan
        assert eight <= ws <= eight + (1 << 30) + (64 << 20), (R, ws, eight)


# one realization in the last pass, whole passes, a ragged last one; items of 4 tiles (enough workgroups
# for them only with the passes counted); very many passes of one item
@pytest.mark.gpu
@pytest.mark.parametrize("B,F,R,L,npar", [(700, 2, 513, 5, 0), (1100, 2, 1024, 1, 0), (2600, 3, 1537, 16, 7),
                                          (2600, 40, 27000, 5, 0), (40, 1, 16780000, 1, 0)])
def test_many_realizations(gpu, B, F, R, L, npar):
    from holodeck_amd import _lib, engine
    from holodeck_amd import device as D
    print(f"[many realizations B={B} F={F} R={R}]", flush=True)
    rng = np.random.default_rng(R)
    lam = 10.0 ** rng.uniform(-2, 7, size=(B, F))      # table-less means among them
    h = 10.0 ** rng.uniform(-12, -9, size=(B, F)) / (1.0 + lam)
    par = D.to_dev(rng.uniform(1.0, 2.0, size=(npar, B, F))) if npar else None
    n_d, h_d = D.to_dev(lam), D.to_dev(h)
    order = engine.order_desc(h_d, col=0)
    rec = torch.empty((B, F, R), dtype=torch.float64, device="cuda")
    got = engine.realize(n_d, h_d, R, L, _lib.HD_SEL_SORTED, order=order, par=par, seed=5, record_counts=rec)
    want = engine.realize(n_d, h_d, R, L, _lib.HD_SEL_SORTED, order=order, par=par, counts=rec)
    assert torch.equal(got[1], want[1]) and torch.equal(got[0], want[0])
    # two sums of 2600 non-negative terms in any order: 2 x 2600 x 2^-53 of the total
    total = want[2] + want[0].sum(dim=2)
    assert bool(((got[2] - want[2]).abs() <= 1e-12 * total).all())
    if npar:
        some = want[2] > 1e-3 * total
        assert bool(((got[3] - want[3]).abs()[:, some] <= 1e-8 * want[3].abs()[:, some]).all())
    # 6 standard errors of the mean, widened for the skewed small means
    assert bool(((rec.mean(dim=2) - n_d).abs() <= 6.0 * torch.sqrt(n_d / R) + 12.0 / R).all())
