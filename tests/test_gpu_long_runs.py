"""Runs of several thousand gates on few qubits, where one qubit with few gates
holds up the others: the gradient and the batched gradient against the
parameter-shift rule and the oracle."""
import math

import pytest

from test_plan_progress import held_up

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,heavy,per", [(6, 5, 1005), (12, 11, 1100), (14, 9, 1100)])
def test_gradients_of_held_up_gates(orc, n, heavy, per):
    print(f"case held up {n} {heavy} {per}", flush=True)
    import spinoza_amd as spz
    from spinoza_amd import _native as N
    from spinoza_amd.autograd import adjoint_gradient, batch_adjoint
    from spinoza_amd.executor import run_ops
    ops = held_up(heavy, per)
    ref = orc.OracleState(n)
    orc.set_threads(16)
    orc.execute(ref, ops)
    e_ref = ref.ising_energy(1.0)
    s = spz.State(n)
    e, g, _ = adjoint_gradient(s, ops, 1.0)
    # every gate adds a few roundings of 1.1e-16 to amplitudes of norm 1, and
    # the energy and its gradients are at most 2 (2 n - 1) times such an error
    tol = 8 * len(ops) * 1.2e-16 * 4 * n
    assert abs(e - e_ref) < tol
    (eb,), (gb,), _ = batch_adjoint([(n, ops)], 1.0, wg_max_qubits=20)
    assert abs(eb - e) < tol and max(abs(g - gb)) < tol
    # a controlled rotation's energy is a0 + a1 cos(t/2 + p1) + a2 cos(t + p2): its
    # derivative from the shifts pi/2 and 3 pi/2
    c1, c2 = (math.sqrt(2) + 1) / (4 * math.sqrt(2)), (math.sqrt(2) - 1) / (4 * math.sqrt(2))
    for i in (1, len(ops) // 2, len(ops) - 2):
        en = []
        for d in (math.pi / 2, -math.pi / 2, 3 * math.pi / 2, -3 * math.pi / 2):
            o = list(ops)
            o[i] = dict(ops[i], theta=ops[i]["theta"] + d)
            t = spz.State(n)
            run_ops(t, o, mode=N.EXEC_PLAIN)
            en.append(spz.ising_energy(t, 1.0))
        assert abs(g[i] - (c1 * (en[0] - en[1]) - c2 * (en[2] - en[3]))) < 4 * tol, i
