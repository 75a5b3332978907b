"""Tile sweeps that store amplitudes away from where they were loaded: X gates
absorbed into the sweep's frame move whole wavefronts' amplitudes to each other's
places.  Every pass has to give the same permutation, bit for bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,n", [("f64", 13), ("f64", 20), ("f64", 24), ("f32", 13),
                                    ("f32", 21), ("f32", 25)])
def test_flipped_stores_wait_for_loads(prec, n):
    import spinoza_amd as spz
    from spinoza_amd import _native as N
    from spinoza_amd.executor import run_ops
    from spinoza_amd.workloads import op
    rng = np.random.default_rng(n)
    re, im = rng.standard_normal(1 << n), rng.standard_normal(1 << n)
    if prec == "f32":
        re, im = re.astype(np.float32).astype(np.float64), im.astype(np.float32).astype(np.float64)
    s = spz.State.from_arrays(re, im, prec)
    for low, high in ((0, 12), (4, 12), (10, 12), (n - 8, n)):
        print(f"case flipped stores {prec} {n} {low}..{high - 1}", flush=True)
        qs = list(range(low, high))
        flip = np.arange(1 << n) ^ sum(1 << q for q in qs)
        for _ in range(5):
            run_ops(s, [op(N.X, q) for q in qs], mode=N.EXEC_AUTO)
            re, im = re[flip], im[flip]
        gr, gi = s.download()
        assert np.array_equal(gr, re) and np.array_equal(gi, im)
