"""Sampling of states with many blocks, whose running sums the host forms (from
24 qubits on), against the oracle, index for index: few and many samples,
several rounds, a single block of weight, a zero state, NaN."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,prec", [(23, "f64"), (24, "f64"), (25, "f32")])
def test_many_blocks_match_oracle(orc, n, prec):
    import spinoza_amd as spz
    print(f"case sample many blocks n={n} {prec}", flush=True)
    ref = orc.random_state(900 + n, n)
    if prec == "f32":
        ref.re[:] = ref.re.astype(np.float32)
        ref.im[:] = ref.im.astype(np.float32)
    s = spz.State.from_arrays(ref.re, ref.im, prec)
    for k in (1, 2000, 20000):  # (from 16384 on samples go through device memory)
        u = orc.uniforms(901 + k, k)
        u[0] = 0.0
        u[-1] = np.nextafter(1.0, 0.0)
        assert np.array_equal(spz.sample(s, u), ref.sample(u)), k
    u = orc.uniforms(77, (1 << 20) + 4321)  # two rounds
    got = spz.sample(s, u)
    parts = [spz.sample(s, u[a:a + 300000]) for a in range(0, len(u), 300000)]
    assert np.array_equal(got, np.concatenate(parts))
    # one NaN amplitude: every sample is the last index of positive weight
    s.upload(np.array([np.nan]), np.array([0.0]), 70000)
    assert set(spz.sample(s, u[:100]).tolist()) == {(1 << n) - 1}


def test_basis_and_zero_states():
    import spinoza_amd as spz
    from spinoza_amd import _native as N
    print("case sample basis and zero", flush=True)
    u = np.array([0.0, 0.5, np.nextafter(1.0, 0.0)])
    s = spz.State(26)
    for index in (0, 4095, 12345678, (1 << 26) - 1):
        s.set_basis(index)
        assert spz.sample(s, u).tolist() == [index] * 3
    s.upload(np.array([0.0]), np.array([0.0]), (1 << 26) - 1)
    with pytest.raises(N.SpinozaError) as err:
        spz.sample(s, u)
    assert err.value.code == N.ERR_PROB
    s.set_basis(7)
    assert spz.sample(s, u).tolist() == [7] * 3
