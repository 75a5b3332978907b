"""Dense blocks at the edges of their kernels, bit for bit against the oracle: one
workgroup of vectors and one vector less, blocks at every offset (runs of memory
and strided), controls below, between a workgroup's vectors and above, both
precisions.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("m", [2, 3, 4, 5])
def test_dense_block_offsets(orc, m, prec):
    import spinoza_amd as spz
    from spinoza_amd import Unitary
    rng = np.random.default_rng(m)
    a = rng.normal(size=(1 << m, 1 << m)) + 1j * rng.normal(size=(1 << m, 1 << m))
    q, _ = np.linalg.qr(a)
    for n in (m + 5, m + 6, 13, 15):
        base = orc.random_state(40 + n, n)
        if prec == "f32":
            base.re[:] = base.re.astype(np.float32)
            base.im[:] = base.im.astype(np.float32)
        for t in range(n - m + 1):
            for c in {-1, 0, t - 1, t + m, n - 1, (t + m + 3) % n}:
                if c != -1 and (not 0 <= c < n or t <= c < t + m):
                    continue
                print(f"case dense rows m={m} n={n} t={t} c={c} {prec}", flush=True)
                ref = base.copy()
                s = spz.State.from_arrays(base.re, base.im, prec)
                if c < 0:
                    ref.transform_u(q, t)
                    spz.transform_u(s, Unitary.from_matrix(q), t)
                else:
                    ref.transform_u(q, t, control=c)
                    spz.c_transform_u(s, Unitary.from_matrix(q), c, t)
                re, im = s.download()
                f = (lambda x: x.astype(np.float32)) if prec == "f32" else (lambda x: x)
                assert np.array_equal(re, f(ref.re)) and np.array_equal(im, f(ref.im))
