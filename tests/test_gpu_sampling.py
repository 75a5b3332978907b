"""Inverse-CDF sampling on the GPU against the oracle, index for index.

The sizes are those where the block structure can go wrong: states smaller
than a block, exactly one, two and many blocks, blocks of weight zero, all
samples in one block, more uniforms than one round takes, and uniforms at the
ends of [0, 1).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def spz():
    import spinoza_amd
    return spinoza_amd


def both(spz, orc, re, im):
    n = int(len(re)).bit_length() - 1
    ref = orc.OracleState(n)
    ref.re[:], ref.im[:] = re, im
    return spz.State.from_arrays(re, im), ref


@pytest.mark.parametrize("n,k", [(1, 3), (5, (1 << 20) + 77), (11, 1000), (12, 1), (13, 4096),
                                 (16, 5000), (20, 4096)])
def test_sample_matches_oracle(spz, orc, n, k):
    print(f"case sample n={n} k={k}", flush=True)
    base = orc.random_state(300 + n, n)
    s, ref = both(spz, orc, base.re, base.im)
    u = orc.uniforms(301 + n, k)
    u[0] = 0.0
    u[-1] = np.nextafter(1.0, 0.0)
    assert np.array_equal(spz.sample(s, u), ref.sample(u))


@pytest.mark.parametrize("where", [[0], [4095, 4096], [12288 + 5, (1 << 15) - 1]])
def test_sample_sparse_states(spz, orc, where):
    """Most blocks have weight zero; every sample falls in the same one or two."""
    print(f"case sample sparse {where}", flush=True)
    re, im = np.zeros(1 << 15), np.zeros(1 << 15)
    for i, j in enumerate(where):
        re[j], im[j] = 0.6 / (i + 1), 0.1
    s, ref = both(spz, orc, re, im)
    u = np.concatenate([[0.0, np.nextafter(1.0, 0.0)], orc.uniforms(9, 3000)])
    got = spz.sample(s, u)
    assert np.array_equal(got, ref.sample(u))
    assert set(got.tolist()) <= set(where)


def test_sample_fp32_state(spz, orc):
    print("case sample f32", flush=True)
    base = orc.random_state(77, 14)
    re, im = base.re.astype(np.float32), base.im.astype(np.float32)
    s = spz.State.from_arrays(re, im, "f32")
    _, ref = both(spz, orc, re.astype(np.float64), im.astype(np.float64))
    u = orc.uniforms(78, 2000)
    assert np.array_equal(spz.sample(s, u), ref.sample(u))


def test_sample_zero_state_is_an_error(spz, orc):
    print("case sample zero state", flush=True)
    z = np.zeros(1 << 13)
    s = spz.State.from_arrays(z, z)
    with pytest.raises(spz.SpinozaError):
        spz.sample(s, np.array([0.3, 0.6]))
    s.set_basis(5000)  # the next call works again
    assert spz.sample(s, np.array([0.1, 0.9])).tolist() == [5000, 5000]
