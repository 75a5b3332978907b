"""Batched gradients at the edges of their sweeps, against the single-circuit
gradient (which the oracle pins): circuits of 1 to 20 qubits in one call, empty
and parameter-free circuits, many gate kinds and controls, several chunks, and
every way to spread a circuit over workgroups.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def spz():
    import spinoza_amd
    return spinoza_amd


def circuit(n, gates, seed):
    from spinoza_amd import _native as N
    from spinoza_amd.workloads import op
    rng = np.random.default_rng(seed)
    ops = []
    for _ in range(gates):
        kind = [N.H, N.X, N.Y, N.Z, N.P, N.RX, N.RY, N.RZ, N.U][int(rng.integers(9))]
        qs = [int(q) for q in rng.permutation(n)]
        o = op(kind, qs[0], theta=rng.uniform(-9, 9), phi=rng.uniform(-4, 4), lam=rng.uniform(-4, 4))
        k = int(rng.integers(0, min(n, 8)))  # 0 to 7 controls
        if rng.random() < 0.4:
            for j, q in enumerate(qs[1:1 + k]):
                o["zeros" if j % 3 == 2 else "ones"] |= 1 << q
        ops.append(o)
    return n, ops


def check(spz, circuits, **opts):
    from spinoza_amd.autograd import adjoint_gradient, batch_adjoint
    energies, grads, stats = batch_adjoint(circuits, 0.8, **opts)
    for (n, ops), e, g in zip(circuits, energies, grads):
        e1, g1, _ = adjoint_gradient(spz.State(n), ops, 0.8)
        assert abs(e - e1) < 1e-12, n
        assert len(g) == len(ops) and (not len(ops) or np.max(np.abs(g - g1)) < 1e-12), n
    return stats


@pytest.mark.parametrize("opts", [{}, {"group_qubits": -1}, {"group_qubits": 8, "wg_per_cu": 1},
                                  {"group_qubits": 13, "wg_per_cu": 2, "use_graph": False}])
def test_batch_of_every_size(spz, opts):
    print(f"case batch sizes {opts}", flush=True)
    circuits = [circuit(n, 3 * n + 5, n) for n in range(1, 21)]
    circuits += [(7, []), circuit(15, 1, 3), (13, [])]
    stats = check(spz, circuits, wg_max_qubits=64, **opts)
    assert stats["n_large"] == 0 and stats["n_small"] == len(circuits)
    gq = {0: 12, -1: 64}.get(opts.get("group_qubits", 0), opts.get("group_qubits", 0))
    assert stats["n_group"] == sum(n > gq for n, _ in circuits)


def test_batch_of_many_chunks(spz):
    """More tiles and more ops than a chunk takes, some circuits above the
    switch point; twice, the second time from kept scratch."""
    print("case batch chunks", flush=True)
    circuits = [circuit(3 + (5 * i) % 14, 40 + i % 90, 100 + i) for i in range(300)]
    for _ in range(2):
        stats = check(spz, circuits, wg_max_qubits=15)
        assert stats["n_large"] == sum(n > 15 for n, _ in circuits) > 0


def test_empty_circuits_are_the_zero_state(spz):
    from spinoza_amd.autograd import batch_adjoint
    print("case batch empty", flush=True)
    e, g, _ = batch_adjoint([(n, []) for n in (1, 5, 12, 14)], 1.0)
    assert e.tolist() == [0.0, 4.0, 11.0, 13.0] and all(len(x) == 0 for x in g)
