"""SWAPs inside tile sweeps, against one launch per gate (which the oracle pins):
random circuits with SWAPs anywhere and of any qubits (low ones, both in the
tile's registers or lanes, far apart, controlled), runs of SWAPs alone, and the
Fourier transform.  Program order is bit-identical; AUTO within the roundings of
its gates.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def circuit(n, gates, seed):
    from spinoza_amd import _native as N
    from spinoza_amd.workloads import op
    rng = np.random.default_rng(seed)
    kinds = [N.H, N.X, N.Y, N.Z, N.P, N.RX, N.RY, N.RZ, N.U]
    ops = []
    for _ in range(gates):
        qs = [int(q) for q in rng.permutation(n)]
        r = rng.random()
        if r < 0.25:
            o = op(N.SWAP, qs[0], t1=qs[1])
            if rng.random() < 0.15:
                o["ones"] = 1 << qs[2]
        else:
            o = op(kinds[int(rng.integers(9))], qs[0], theta=rng.uniform(-6, 6),
                   phi=rng.uniform(-4, 4), lam=rng.uniform(-4, 4))
            if r < 0.6:
                o["ones" if rng.random() < 0.7 else "zeros"] |= 1 << qs[1]
        ops.append(o)
    return ops


def both(n, prec, ops, mode):
    import spinoza_amd as spz
    from spinoza_amd import _native as N
    from spinoza_amd.executor import run_ops
    from spinoza_amd.workloads import op
    rng = np.random.default_rng(n)
    start = [op(N.RY, q, theta=rng.uniform(-3, 3)) for q in range(n)]
    start += [op(N.P, q, theta=rng.uniform(-3, 3), ones=1 << ((q + 5) % n)) for q in range(n)]
    out = []
    for m in (N.EXEC_PLAIN, mode):
        s = spz.State(n, prec)
        run_ops(s, start, mode=N.EXEC_PLAIN)
        run_ops(s, ops, mode=m)
        out.append(s.to_numpy())
    return out


@pytest.mark.parametrize("n,gates", [(13, 60), (14, 120), (17, 200), (20, 200), (23, 120)])
def test_swaps_in_sweeps(n, gates):
    from spinoza_amd import _native as N
    for seed in range(4):
        ops = circuit(n, gates, 100 * n + seed)
        print(f"case swaps n={n} seed={seed}", flush=True)
        want, got = both(n, "f64", ops, N.EXEC_STRICT)
        assert np.array_equal(want, got)
        want, got = both(n, "f64", ops, N.EXEC_AUTO)
        # at most 16 roundings of an amplitude per gate on either side
        assert np.linalg.norm(got - want) <= 32 * gates * 2.0 ** -53 * np.linalg.norm(want)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n", [13, 16, 21])
def test_swaps_alone(n, prec):
    from spinoza_amd import _native as N
    from spinoza_amd.workloads import op
    rng = np.random.default_rng(7 * n)
    for count in (1, 2, 3, n // 2, 3 * n):
        print(f"case swaps alone n={n} {prec} {count}", flush=True)
        ops = [op(N.SWAP, int(a), t1=int(b))
               for a, b in (rng.choice(n, 2, replace=False) for _ in range(count))]
        want, got = both(n, prec, ops, N.EXEC_AUTO)
        assert np.array_equal(want, got)


@pytest.mark.parametrize("n", [13, 18, 22])
def test_fourier_transform(n):
    from spinoza_amd import _native as N
    from spinoza_amd.workloads import qft
    print(f"case qft n={n}", flush=True)
    ops = qft(n)
    want, got = both(n, "f64", ops, N.EXEC_AUTO)
    assert np.linalg.norm(got - want) <= 32 * len(ops) * 2.0 ** -53 * np.linalg.norm(want)
    want, got = both(n, "f32", ops, N.EXEC_AUTO)
    assert np.linalg.norm(got - want) <= 32 * len(ops) * 2.0 ** -24 * np.linalg.norm(want)
