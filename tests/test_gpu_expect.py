"""Expectations of many qubits in one call, and the Ising energy, against the
oracle bit for bit.

Sizes around the reduction block (4096 amplitudes): below it, one, two, eight
and more blocks; targets in every class the block kernel tells apart (in the
wavefront, across wavefronts, in registers, in other blocks), repeated, in any
order, and more of them than one pass or one round of results takes.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def spz():
    import spinoza_amd
    return spinoza_amd


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("n", [3, 11, 12, 13, 15, 17])
def test_expectations_of_all_targets(spz, orc, n, precision):
    print(f"case expect n={n} {precision}", flush=True)
    base = orc.random_state(400 + n, n)
    if precision == "f32":
        base.re[:] = base.re.astype(np.float32)
        base.im[:] = base.im.astype(np.float32)
    s = spz.State.from_arrays(base.re, base.im, precision)
    rng = np.random.default_rng(n)
    lists = [list(range(n)), [n - 1], list(rng.integers(0, n, size=131)), []]
    for obs in "xyz":
        ref = [base.xyz_expectation_value(obs, [t])[0] for t in range(n)]
        for targets in lists:
            got = spz.xyz_expectation_value(obs, s, targets)
            assert got == [ref[t] for t in targets], (obs, targets)
    for hx in (1.0, -0.3):
        assert spz.ising_energy(s, hx) == base.ising_energy(hx)
    with pytest.raises(spz.SpinozaError):
        spz.xyz_expectation_value("x", s, [0, n])


def test_expectations_keep_infinities_and_nan_apart(spz, orc):
    """A NaN amplitude makes every sum NaN; an infinite one is not hidden."""
    print("case expect nan/inf", flush=True)
    for bad in (np.nan, np.inf):
        base = orc.random_state(5, 13)
        base.re[4100] = bad
        s = spz.State.from_arrays(base.re, base.im)
        for obs in "xyz":
            got = spz.xyz_expectation_value(obs, s, [0, 7, 9, 12])
            ref = base.xyz_expectation_value(obs, [0, 7, 9, 12])
            np.testing.assert_array_equal(np.isfinite(got), np.isfinite(ref))
