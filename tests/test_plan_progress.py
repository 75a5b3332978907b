"""Host-side tests of planning (no GPU needed): every plan makes progress and
holds each gate once, also where one qubit with few gates holds up more than a
thousand gates on each of the others."""
import ctypes

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


def chip_plan(n, ops, reverse):
    """The plan of batched circuits and of states of at most 12 qubits
    (spz::chip_plan, an inner function of the library): the gates of its program."""
    f = N.lib()._ZN3spz9chip_planEiPK6spz_opmbRNS_8ChipPlanE
    f.argtypes = [ctypes.c_int, ctypes.c_void_p, ctypes.c_uint64, ctypes.c_bool, ctypes.c_void_p]
    arr, keep = encode_ops(ops)
    plan = (ctypes.c_uint64 * 9)()  # three empty std::vector: program, sweeps, gradients
    rc = f(n, ctypes.addressof(arr), len(ops), reverse, ctypes.addressof(plan))
    del keep
    if rc:
        raise N.SpinozaError(rc, N.lib().spz_last_error().decode())
    raw = ctypes.string_at(plan[0], plan[1] - plan[0])
    types = np.frombuffer(raw, dtype=np.int32).reshape(-1, TILE_OP // 4)[:, 0]
    return int(np.sum(types != LAYOUT))


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
