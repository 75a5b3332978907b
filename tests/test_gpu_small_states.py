"""States of at most 12 qubits, which run a whole circuit (and its reverse
sweep) in one launch: amplitudes bit-identical to the oracle in AUTO and
STRICT, for every size from 1 to 12 qubits; FP32 storage within its rounding
of one launch per gate; gradients against oracle parameter shift.
"""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def spz():
    import spinoza_amd
    return spinoza_amd


def circuit(n, seed):
    """Every gate kind, 1- and 0-controls, SWAPs, noise on both sides of its draw."""
    from spinoza_amd import _native as N
    from spinoza_amd.workloads import op
    rng = np.random.default_rng(seed)
    ops = []
    for i in range(6 * n + 6):
        kind = [N.H, N.X, N.Y, N.Z, N.P, N.RX, N.RY, N.RZ, N.U][int(rng.integers(9))]
        qs = [int(q) for q in rng.permutation(n)]
        o = op(kind, qs[0], theta=rng.uniform(-9, 9), phi=rng.uniform(-4, 4), lam=rng.uniform(-4, 4))
        if n > 1 and i % 3 == 1:
            o["ones"] = 1 << qs[1]
        if n > 2 and i % 4 == 2:
            o["zeros"] = 1 << qs[2]
        ops.append(o)
        if n > 1 and i % 5 == 0:
            ops.append(op(N.SWAP, qs[0], t1=qs[1]))
        if i % 7 == 3:
            ops.append(dict(op(N.BITFLIP, qs[0], theta=0.5), u=[0.2, 0.8][i & 1]))
    return ops


@pytest.mark.parametrize("n", range(1, 13))
def test_small_states_bit_identical(spz, orc, n):
    print(f"case small n={n}", flush=True)
    from spinoza_amd import _native as N
    from spinoza_amd.executor import run_ops
    ops = circuit(n, n)
    base = orc.random_state(500 + n, n)
    ref = base.copy()
    orc.execute(ref, ops)
    for mode in (N.EXEC_AUTO, N.EXEC_STRICT, N.EXEC_PLAIN):
        s = spz.State.from_arrays(base.re, base.im)
        run_ops(s, ops, mode=mode)
        re, im = s.download()
        assert np.array_equal(re, ref.re) and np.array_equal(im, ref.im), mode
    a, b = (spz.State.from_arrays(base.re, base.im, "f32") for _ in range(2))
    run_ops(a, ops, mode=N.EXEC_AUTO)
    run_ops(b, ops, mode=N.EXEC_PLAIN)
    # PLAIN rounds to FP32 after every gate, at most 2^-24 of an amplitude each
    tol = len(ops) * 2.0 ** -23
    for x, y in zip(a.download(), b.download()):
        assert np.max(np.abs(x - y)) < tol


def test_small_states_with_measurement_and_blocks(spz, orc):
    """Runs end at measurements and dense blocks; classical controls after them."""
    print("case small measured", flush=True)
    from spinoza_amd import _native as N
    from spinoza_amd.executor import run_ops
    from spinoza_amd.workloads import op
    n = 6
    ops = circuit(n, 3) + [dict(op(N.M, 2), u=0.4)]
    ops += [op(N.X, 4, ones=1 << 2, classical=True), op(N.H, 0),
            op(N.SWAP, 1, t1=3, ones=1 << 2, classical=True)]
    ops += circuit(n, 4)
    s, p = spz.State(n), spz.State(n)
    assert run_ops(s, ops) == run_ops(p, ops, mode=N.EXEC_PLAIN)
    for x, y in zip(s.download(), p.download()):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("n,ckpt", [(1, 0), (2, 1), (5, 4), (8, 0), (12, 25)])
def test_small_gradients_vs_parameter_shift(spz, orc, n, ckpt):
    print(f"case small gradient n={n}", flush=True)
    from spinoza_amd import _native as N
    from spinoza_amd.autograd import adjoint_gradient
    from spinoza_amd.workloads import op
    rng = np.random.default_rng(n)
    ops = []
    for layer in range(8):  # more than 64 parameters at 12 qubits
        for q in range(n):
            ops.append(op(N.H, q))
            ops.append(op([N.RX, N.RY, N.RZ, N.P][(q + layer) % 4], q, theta=rng.uniform(-7, 7)))
        if n > 1:
            ops.append(op(N.SWAP, layer % n, t1=(layer + 1) % n))
            ops.append(op(N.X, (layer + 1) % n, ones=1 << (layer % n)))

    def energy(o):
        st = orc.OracleState(n)
        orc.execute(st, o)
        return st.ising_energy(0.9)

    s = spz.State(n)
    e, g, drift = adjoint_gradient(s, ops, 0.9, ckpt)
    assert abs(e - energy(ops)) < 1e-12 and drift < 1e-13
    params = [i for i, o in enumerate(ops) if o["kind"] in (N.RX, N.RY, N.RZ, N.P)]
    assert all(g[i] == 0.0 for i in range(len(ops)) if i not in params)
    for i in params[:: max(1, len(params) // 16)]:
        v = []
        for sg in (1.0, -1.0):
            o = [dict(x) for x in ops]
            o[i]["theta"] += sg * math.pi / 2
            v.append(energy(o))
        assert abs(g[i] - 0.5 * (v[0] - v[1])) < 1e-10
