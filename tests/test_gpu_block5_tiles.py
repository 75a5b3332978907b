"""Dense 5-qubit blocks at the edges of their kernel, against gate by gate
execution (which the oracle pins): one tile, as many tiles as workgroups and
several tiles per workgroup, with none to all of the line's low qubits in the
block (both ways the results are stored), in any order of qubits.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# n 12: one tile; 20 (FP64) and 21 (FP32): a tile per workgroup of 256 CUs
SIZES = [("f64", 12), ("f64", 20), ("f64", 22), ("f32", 12), ("f32", 21), ("f32", 23)]


def block(N, op, rng, q):
    """16 gates that fall into one block on the qubits q."""
    ops = [op(N.RX, x, theta=rng.uniform(-4, 4)) for x in q]
    ops += [op(N.U, x, theta=rng.uniform(-4, 4), phi=rng.uniform(-4, 4),
               lam=rng.uniform(-4, 4)) for x in q]
    ops += [op(N.RY, q[j], theta=rng.uniform(-4, 4), ones=1 << q[j - 1]) for j in range(5)]
    return ops + [op(N.P, q[0], theta=0.7, zeros=1 << q[3])]


@pytest.mark.parametrize("prec,n", SIZES)
def test_block5_tiles(prec, n):
    import spinoza_amd as spz
    from spinoza_amd import _native as N
    from spinoza_amd.executor import run_ops
    from spinoza_amd.workloads import op
    rng = np.random.default_rng(n)
    start = [op(N.RY, x, theta=rng.uniform(-2, 2)) for x in range(n)]
    start += [op(N.P, x, theta=rng.uniform(-2, 2), ones=1 << ((x + 1) % n)) for x in range(n)]
    # 16 gates put 16 * 8 roundings into each of 32 columns of U, the product 64
    # into each row of norm sqrt(64): (16 * 8 * sqrt(32) + 64 * sqrt(64)) u, and
    # 4 per gate on the other side
    u = 2.0 ** (-53 if prec == "f64" else -24)
    bound = (16 * 8 * 32 ** 0.5 + 64 * 8 + 4 * 16) * u
    for q in ([0, 1, 2, 3, 4], [4, n - 1, 0, 2, 1], [n - 2, 3, 1, n - 4, 0], [2, n - 1, 6, 0, 8],
              [n - 3, 1, 10, 5, 7], [n - 1, n - 2, n - 3, n - 4, n - 5], [4, 11, 9, 6, 5]):
        print(f"case block5 {prec} {n} {q}", flush=True)
        ops = block(N, op, rng, q)
        want, got = spz.State(n, prec), spz.State(n, prec)
        run_ops(want, start, mode=N.EXEC_PLAIN)
        run_ops(got, start, mode=N.EXEC_PLAIN)
        run_ops(want, ops, mode=N.EXEC_PLAIN)
        run_ops(got, ops, mode=N.EXEC_DENSE5)
        w = want.to_numpy().astype(np.complex128)
        g = got.to_numpy().astype(np.complex128)
        assert np.linalg.norm(g - w) <= bound * np.linalg.norm(w)
