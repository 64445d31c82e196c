"""hd_order_desc where its path changes: one workgroup up to a tile of 4096 keys, tiles above; few and
many equal keys, keys that differ in single digits, signed zeros and infinities, against numpy's stable
sort (exact)."""
import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("B,stride", [(1, 1), (2, 3), (63, 1), (65, 2), (255, 1), (257, 1), (1023, 1), (4095, 1), (4096, 5),
                                      (4097, 1), (8192, 1), (8193, 3), (262143, 1), (262145, 1), (300001, 2)])
def test_order_desc_equals_a_stable_sort(gpu, B, stride):
    from holodeck_amd import device as D, engine
    rng = np.random.default_rng(B)
    wide = 10.0 ** rng.uniform(-300, 300, size=B) * rng.choice([-1.0, 1.0], size=B)
    few = rng.integers(0, 5, size=B).astype(float)
    last = (np.full(B, np.float64(1.0)).view(np.int64) + rng.integers(0, 300, size=B)).view(np.float64)   # low digits only
    strain = np.where(rng.random(B) < 0.4, 0.0, 10.0 ** rng.uniform(-40, -30, size=B))
    odd = rng.choice([0.0, -0.0, np.inf, -np.inf, 5e-324, -5e-324, 1.0], size=B)
    for name, key in (("wide", wide), ("few", few), ("last", last), ("strain", strain), ("odd", odd), ("equal", np.ones(B))):
        print(f"[order B={B} stride={stride} {name}]", flush=True)
        grid = rng.random((B, stride))
        grid[:, stride - 1] = key
        got = D.to_host(engine.order_desc(D.to_dev(grid), col=stride - 1))
        assert np.array_equal(got, np.argsort(-key, kind='stable'))
