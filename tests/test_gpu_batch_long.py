"""Batches of long circuits: they run side by side, not one after another, with
the gradients of the single-circuit path."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_long_circuits_share_a_chunk():
    import spinoza_amd as spz
    from spinoza_amd import _native as N
    from spinoza_amd.autograd import adjoint_gradient, batch_adjoint
    from spinoza_amd.workloads import op
    print("case long batch", flush=True)
    circuits = []
    for c in range(24):
        rng = np.random.default_rng(c)
        n, ops = 8 + c % 3, []
        for _ in range(4000):
            a, b = (int(q) for q in rng.permutation(n)[:2])
            kind = [N.RX, N.RY, N.RZ, N.X][int(rng.integers(4))]
            ops.append(op(kind, a, theta=rng.uniform(-3, 3), ones=1 << b if kind == N.X else 0))
        circuits.append((n, ops))
    batch_adjoint(circuits, 1.0, wg_max_qubits=20)
    e, g, st = batch_adjoint(circuits, 1.0, wg_max_qubits=20)
    for (n, ops), x, y in list(zip(circuits, e, g))[::9]:
        e1, g1, _ = adjoint_gradient(spz.State(n), ops, 1.0)
        tol = 8 * len(ops) * 1.2e-16 * 4 * n  # a few roundings a gate, energies up to 2 n
        assert abs(x - e1) < tol and np.max(np.abs(y - g1)) < tol
    # a circuit's time is its chunk's: 24 chunks one after another took 24 of them
    assert st["total_ms"] < 8 * st["p50_ms"], st
