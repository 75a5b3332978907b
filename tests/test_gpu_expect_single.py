"""Single-target expectations (a launch of their own) and the sides of a pair
of blocks that form their common sum: every target alone and with others, bit
for bit the same, and against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n", [12, 13, 14, 15, 18])
def test_single_targets(orc, n, prec):
    import spinoza_amd as spz
    print(f"case single targets n={n} {prec}", flush=True)
    base = orc.random_state(60 + n, n)
    if prec == "f32":
        base.re[:] = base.re.astype(np.float32)
        base.im[:] = base.im.astype(np.float32)
    s = spz.State.from_arrays(base.re, base.im, prec)
    for ob in "xyz":
        alone = [spz.xyz_expectation_value(ob, s, [q])[0] for q in range(n)]
        assert alone == base.xyz_expectation_value(ob, list(range(n)))
        assert spz.xyz_expectation_value(ob, s, list(range(n))) == alone
        assert spz.xyz_expectation_value(ob, s, [n - 1, 0, n - 1]) == [alone[n - 1], alone[0],
                                                                        alone[n - 1]]
