"""The switch point of batched gradients: only sizes that can run batched set it."""
import pytest

pytestmark = pytest.mark.gpu


def test_large_circuits_leave_the_switch_point():
    from spinoza_amd import _native as N
    from spinoza_amd.autograd import batch_autotune
    from spinoza_amd.workloads import hea, op
    print("case autotune", flush=True)
    small = [(n, hea(n, 2, seed=n)[0]) for n in (5, 8, 8, 9)]
    large = [(n, hea(n, 1, seed=n)[0]) for n in (21, 22)]
    point = batch_autotune(small)
    assert point in (5, 8, 9)
    assert batch_autotune(large) == point
    assert batch_autotune(small + large) <= 9
    for bad in ((31, []), (21, [op(N.X, 20, ones=0xFF)]), (22, [op(N.M, 0)])):
        with pytest.raises(N.SpinozaError):
            batch_autotune(small + [bad])
