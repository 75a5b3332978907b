"""Sweeps and gradients for every setting of the number of lowest qubits kept
in the tile (SPZ_TILE_KLO), also outside its range."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("klo", [-3, 0, 1, 8, 9, 11, 12, 40])
def test_gradient_for_every_number_of_low_qubits(monkeypatch, klo):
    print(f"case low qubits {klo}", flush=True)
    import spinoza_amd as spz
    from spinoza_amd import _native as N
    from spinoza_amd.autograd import adjoint_gradient
    from spinoza_amd.executor import run_ops
    from spinoza_amd.workloads import random_circuit
    n = 15
    ops = random_circuit(n, 4, 3)
    plain = spz.State(n)
    run_ops(plain, ops, mode=N.EXEC_PLAIN)
    e0, g0, _ = adjoint_gradient(spz.State(n), ops, 0.7)
    monkeypatch.setenv("SPZ_TILE_KLO", str(klo))
    s = spz.State(n)
    e, g, drift = adjoint_gradient(s, ops, 0.7, 25)
    assert abs(e - e0) < 1e-12 and np.max(np.abs(g - g0)) < 1e-12 and drift < 1e-13
    for a, b in zip(s.download(), plain.download()):
        assert np.max(np.abs(a - b)) < 1e-13
