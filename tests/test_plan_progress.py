"""Host-side tests of planning (no GPU needed): every plan makes progress and
holds each gate once, also where one qubit with few gates holds up more than a
thousand gates on each of the others."""
import ctypes
import time

import numpy as np
import pytest

from spinoza_amd import _native as N
from spinoza_amd.executor import encode_ops, plan_stats
from spinoza_amd.workloads import op

LAYOUT, TILE_OP = 2, 128  # TileOp::type of a layout change; bytes of a TileOp


def held_up(heavy, per):
    """H on qubit 0, `per` rotations controlled by it on each of `heavy` others, H."""
    ops = [op(N.RX, q, theta=0.01 * q + 1e-4 * i, ones=1)
           for q in range(1, heavy + 1) for i in range(per)]
    return [op(N.H, 0)] + ops + [op(N.H, 0)]


def planned(fn, n, ops, *args):
    """The gates in the program that an inner planning function of the library makes."""
    arr, keep = encode_ops(ops)
    plan = (ctypes.c_uint64 * 9)()  # three empty std::vector: program, sweeps, gradients
    rc = fn(ctypes.c_int(n), arr, *args, plan)
    del keep
    if rc:
        raise N.SpinozaError(rc, N.lib().spz_last_error().decode())
    raw = ctypes.string_at(plan[0], plan[1] - plan[0])
    types = np.frombuffer(raw, dtype=np.int32).reshape(-1, TILE_OP // 4)[:, 0]
    return int(np.sum(types != LAYOUT))


def chip_plan(n, ops, reverse):
    """Batched circuits, forward or reverse (spz::chip_plan)."""
    return planned(N.lib()._ZN3spz9chip_planEiPK6spz_opmbRNS_8ChipPlanE, n, ops,
                   ctypes.c_uint64(len(ops)), ctypes.c_bool(reverse))


def adjoint_plan(n, ops):
    """The reverse sweeps of one gradient (spz::adjoint_plan)."""
    return planned(N.lib()._ZN3spz12adjoint_planEiPK6spz_opmmRNS_8ChipPlanE, n, ops,
                   ctypes.c_uint64(0), ctypes.c_uint64(len(ops)))


@pytest.mark.parametrize("reverse", [False, True])
@pytest.mark.parametrize("n,heavy,per", [(5, 4, 1100), (6, 5, 1005), (12, 11, 1100), (13, 12, 1100),
                                         (16, 15, 1100), (20, 5, 3000)])
def test_batched_plans_of_held_up_gates(n, heavy, per, reverse):
    ops = held_up(heavy, per)
    assert chip_plan(n, ops, reverse) == len(ops)


@pytest.mark.parametrize("mode", [N.EXEC_AUTO, N.EXEC_STRICT])
@pytest.mark.parametrize("n,heavy,per", [(13, 12, 1100), (16, 15, 1100), (16, 8, 2500), (20, 3, 1200)])
def test_tile_plans_of_held_up_gates(n, heavy, per, mode):
    ops = held_up(heavy, per)
    st = plan_stats(n, ops, mode=mode)
    assert st["tile_gates"] + st["plain_gates"] == len(ops)


@pytest.mark.parametrize("n,heavy,per", [(6, 5, 1005), (13, 12, 1100), (16, 15, 1100), (20, 3, 1200)])
def test_reverse_plans_of_held_up_gates(n, heavy, per):
    ops = held_up(heavy, per)
    assert adjoint_plan(n, ops) == len(ops)


@pytest.mark.parametrize("klo", [-3, 0, 1, 8, 9, 11, 12, 13, 40])
def test_plans_for_every_number_of_low_qubits(monkeypatch, klo):
    """SPZ_TILE_KLO outside its range counts as the nearest number in it; a
    reverse sweep always has room for a gate on any qubit."""
    monkeypatch.setenv("SPZ_TILE_KLO", str(klo))
    ops = [op([N.RX, N.RZ, N.H][q % 3], q, theta=0.1 * q, ones=1 << ((q + 5) % 18))
           for r in range(3) for q in range(18)]
    swaps = [op(N.SWAP, q, t1=17 - q) for q in range(9)]
    assert adjoint_plan(18, ops + swaps) == len(ops) + 3 * len(swaps)
    st = plan_stats(18, ops + swaps)
    assert st["tile_gates"] + st["plain_gates"] == len(ops) + len(swaps)


@pytest.mark.parametrize("reverse", [False, True])
def test_batched_planning_time_is_linear(reverse):
    """Four times the gates of a 10-qubit circuit: 4 times the time where a sweep
    has a bounded number of gates, 16 times where a circuit is one sweep."""
    rng = np.random.default_rng(3)
    ops = []
    for _ in range(24000):
        a, b = (int(q) for q in rng.permutation(10)[:2])
        kind = [N.RX, N.RY, N.RZ, N.X][int(rng.integers(4))]
        ops.append(op(kind, a, theta=0.1, ones=1 << b if kind == N.X else 0))
    took = []
    for part in (ops[:6000], ops):
        best = float("inf")
        for _ in range(3):
            t = time.process_time()
            assert chip_plan(10, part, reverse) == len(part)
            best = min(best, time.process_time() - t)
        took.append(best)
    assert took[1] < 8 * took[0], took
