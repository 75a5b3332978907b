"""Host-only: which runs of a small state go op by op."""
import numpy as np
import pytest

from spinoza_amd import _native as N
from spinoza_amd.executor import plan_stats
from spinoza_amd.workloads import op


def short_run(n, length, seed):
    """`length` ops: gates with 0- and 1-controls, SWAPs, noise that flips."""
    rng = np.random.default_rng(seed)
    ops = []
    for i in range(length):
        qs = [int(q) for q in rng.permutation(n)]
        o = op([N.H, N.RX, N.U, N.P, N.Y][i % 5], qs[0], theta=rng.uniform(-5, 5), phi=0.3, lam=-1.2)
        if n > 2 and i % 3 == 1:
            o = op(N.SWAP, qs[0], t1=qs[1], ones=(1 << qs[2]) * (i & 1))
        elif n > 1 and i % 2:
            o["zeros" if i % 4 == 3 else "ones"] = 1 << qs[1]
        elif i % 7 == 6:
            o = dict(op(N.BITFLIP, qs[0], theta=0.5), u=0.25)
        ops.append(o)
    return ops


@pytest.mark.parametrize("mode", [N.EXEC_AUTO, N.EXEC_STRICT])
@pytest.mark.parametrize("n", [3, 12])
def test_short_runs_go_op_by_op(n, mode):
    for length in range(1, 12):
        st = plan_stats(n, short_run(n, length, length), mode=mode)
        if length <= 5:
            assert st["plain_gates"] == length and st["sweeps"] == 0
        else:
            assert st["plain_gates"] == 0 and st["sweeps"] == 1
