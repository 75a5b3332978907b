"""Reverse tile sweeps of the adjoint gradient (states of more than 12 qubits)
at their edges: two and four tiles, more gradients than one sweep takes,
sweeps of a single gate, controls inside and outside the tile, controlled
SWAPs, FP32 storage.  Gradients against oracle parameter shift (exact for
uncontrolled RX, RY, RZ and P), the final state against the oracle.
"""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def spz():
    import spinoza_amd
    return spinoza_amd


def final(orc, n, ops):
    """The oracle's final state; a controlled SWAP, which the oracle has not,
    as three controlled X."""
    from spinoza_amd import _native as N
    from spinoza_amd.workloads import op
    flat = []
    for o in ops:
        if o["kind"] == N.SWAP and (o["ones"] or o["zeros"]):
            a, b = o["target"], o["t1"]
            flat += [op(N.X, a, ones=1 << b),
                     op(N.X, b, ones=o["ones"] | 1 << a, zeros=o["zeros"]),
                     op(N.X, a, ones=1 << b)]
        else:
            flat.append(o)
    s = orc.OracleState(n)
    orc.execute(s, flat)
    return s


def energy(orc, n, ops):
    return final(orc, n, ops).ising_energy(1.0)


def shift(orc, n, ops, i):
    e = []
    for sg in (1.0, -1.0):
        o = [dict(x) for x in ops]
        o[i]["theta"] += sg * math.pi / 2
        e.append(energy(orc, n, o))
    return 0.5 * (e[0] - e[1])


def circuits(n, name):
    from spinoza_amd import _native as N
    from spinoza_amd.workloads import op
    rng = np.random.default_rng(17)
    ang = lambda: rng.uniform(-7.0, 7.0)
    ops = [op(N.H, q) for q in range(n)]
    if name == "single":  # one gate in the whole reverse sweep of a segment
        return [op(N.RY, n - 1, theta=2.5)]
    if name == "many":  # 5 n diagonal gates and a rotation layer: over 64 gradients in one tile
        for r in range(5):
            for q in range(n):
                ops.append(op([N.RZ, N.P][(q + r) & 1], q, theta=ang()))
        ops += [op(N.RX, q, theta=ang()) for q in range(n)]
        return ops
    for q in range(n):
        ops.append(op([N.RX, N.RY, N.RZ, N.P][q % 4], q, theta=ang()))
        ops.append(op(N.SWAP, q, t1=(q + 3) % n, ones=(1 << ((q + 5) % n)) if q % 3 == 0 else 0,
                      zeros=(1 << ((q + 7) % n)) if q % 4 == 1 else 0))
        ops.append(op([N.X, N.Z, N.Y, N.H, N.U][q % 5], (q + 1) % n, theta=0.4, phi=1.1, lam=-0.6,
                      ones=1 << ((q + 6) % n), zeros=1 << ((q + 9) % n)))
        ops.append(op([N.RY, N.RX][q % 2], q, theta=ang()))
    return ops


@pytest.mark.parametrize("n,name,ckpt", [(13, "mixed", 0), (13, "many", 0), (13, "single", 1),
                                         (14, "mixed", 7), (14, "many", 33)])
def test_reverse_sweeps_vs_parameter_shift(spz, orc, n, name, ckpt):
    print(f"case reverse sweeps {n} {name} {ckpt}", flush=True)
    from spinoza_amd import _native as N
    from spinoza_amd.autograd import adjoint_gradient
    orc.set_threads(16)
    ops = circuits(n, name)
    s = spz.State(n)
    e, g, drift = adjoint_gradient(s, ops, 1.0, ckpt)
    assert drift < 1e-13
    assert abs(e - energy(orc, n, ops)) < 1e-12
    ref = final(orc, n, ops)
    re, im = s.download()
    assert max(np.max(np.abs(re - ref.re)), np.max(np.abs(im - ref.im))) < 1e-12
    params = [i for i, o in enumerate(ops) if o["kind"] in (N.RX, N.RY, N.RZ, N.P)]
    assert all(g[i] == 0.0 for i in range(len(ops)) if i not in params)
    for i in params[:: max(1, len(params) // 24)]:
        assert abs(g[i] - shift(orc, n, ops, i)) < 1e-10, (i, ops[i])
    e32, g32, _ = adjoint_gradient(spz.State(n, "f32"), ops, 1.0, ckpt)
    assert abs(e32 - e) < 1e-4 and np.max(np.abs(g32 - g)) < 1e-4


def test_many_checkpoint_states_are_given_back(spz):
    """Checkpoint states are kept between calls of one shape; another shape
    and another count still give the same gradients."""
    print("case checkpoint pool", flush=True)
    from spinoza_amd.autograd import adjoint_gradient
    from spinoza_amd.workloads import hea
    for n, prec, ck in ((13, "f64", 5), (14, "f64", 11), (13, "f32", 5), (13, "f64", 40), (13, "f64", 3)):
        ops, _, _ = hea(n, 2, seed=n)
        e0, g0, _ = adjoint_gradient(spz.State(n, prec), ops, 1.0, 0)
        e1, g1, drift = adjoint_gradient(spz.State(n, prec), ops, 1.0, ck)
        tol = 1e-12 if prec == "f64" else 1e-4
        assert abs(e0 - e1) < tol and np.max(np.abs(g0 - g1)) < tol and drift < tol
