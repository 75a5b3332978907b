"""Failed device allocations: scratch kept by finished calls is given back and
the allocation tried again; a second failure raises, and the calls after it
are right.  Failures are counted down by the library, no memory is filled."""
import ctypes
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture
def failures():
    from spinoza_amd import _native as N
    c = ctypes.c_int.in_dll(N.lib(), "_ZN3spz16g_alloc_failuresE")
    yield c
    c.value = 0


def free_bytes():
    from spinoza_amd import _native as N
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    N.check(N.lib().spz_sync())
    assert N.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def gradient(n, every, failures=None, count=0):
    """With `every` checkpoints; `count` allocations fail once the state is there."""
    import spinoza_amd as spz
    from spinoza_amd.autograd import adjoint_gradient
    from spinoza_amd.workloads import hea
    ops = hea(n, 2, seed=n)[0]
    s = spz.State(n)
    if failures is not None:
        failures.value = count
    e, g, drift = adjoint_gradient(s, ops, 1.0, len(ops) // every if every else 0)
    return e, g.tobytes(), drift


def batch():
    from spinoza_amd.autograd import batch_adjoint
    from spinoza_amd.workloads import hea
    e, g, _ = batch_adjoint([(16, hea(16, 2, seed=s)[0]) for s in range(6)], 1.0, wg_max_qubits=20)
    return e.tobytes(), [x.tobytes() for x in g]


def test_kept_memory_is_given_back(failures):
    import spinoza_amd as spz
    print("case kept memory", flush=True)
    g0, b0 = gradient(22, 8), batch()
    kept = free_bytes()
    failures.value = 1
    s = spz.State(5)  # its first allocation fails once
    assert failures.value == 0
    # eight checkpoint states, psi and lambda of 64 MiB each
    assert free_bytes() - kept >= 10 * (64 << 20)
    assert abs(s.norm() - 1.0) < 1e-15
    assert gradient(22, 8) == g0 and batch() == b0


def test_failures_inside_calls(failures):
    print("case failures inside calls", flush=True)
    import spinoza_amd as spz
    from spinoza_amd import _native as N
    ref = {n: gradient(n, 5) for n in (18, 19, 20)}
    b0 = batch()
    for n in (18, 20, 19):  # checkpoint states of another shape: allocated in the call
        assert batch() == b0
        assert gradient(n, 5, failures, 1) == ref[n] and failures.value == 0
    with pytest.raises(N.SpinozaError) as err:
        failures.value = 2
        spz.State(20)
    assert err.value.code == N.ERR_OOM
    failures.value = 0
    gradient(18, 0)
    with pytest.raises(N.SpinozaError) as err:
        gradient(20, 5, failures, 100)
    assert err.value.code == N.ERR_OOM
    failures.value = 0
    assert gradient(20, 5) == ref[20] and gradient(18, 5) == ref[18] and batch() == b0


REDUCTION = """
import ctypes
import spinoza_amd as spz
from spinoza_amd import _native as N
failures = ctypes.c_int.in_dll(N.lib(), "_ZN3spz16g_alloc_failuresE")
small, large = spz.State(13), spz.State(26)
want = small.norm()  # the smallest scratch
failures.value = 2
try:
    spz.xyz_expectation_value("z", large, list(range(8)))
    raise SystemExit("no error")
except N.SpinozaError as e:
    assert e.code == N.ERR_OOM, e
failures.value = 0
assert small.norm() == want == 1.0
assert spz.xyz_expectation_value("z", large, list(range(8))) == [1.0] * 8
"""


def test_reduction_scratch_after_a_failure():
    """The scratch of reductions is freed before it grows: after a failure it
    has no size left (a process of its own, where it is still small)."""
    print("case reduction scratch", flush=True)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", REDUCTION], cwd=root, capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
