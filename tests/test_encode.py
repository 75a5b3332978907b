"""Op dicts to C records (the CPython extension behind executor.encode_ops)
against a field-by-field encoding; host only."""
import collections
import types

import numpy as np
import pytest


def field_by_field(N, ops):
    arr = (N.Op_t * max(len(ops), 1))()
    for o, d in zip(arr, ops):
        o.kind, o.target, o.t1 = int(d["kind"]), int(d.get("target", 0)), int(d.get("t1", 0))
        o.theta, o.phi = float(d.get("theta", 0.0)), float(d.get("phi", 0.0))
        o.lam, o.u = float(d.get("lam", 0.0)), float(d.get("u", 1.0))
        o.flags = N.OPF_CLASSICAL if d.get("classical") else 0
        o.ones, o.zeros = int(d.get("ones", 0)), int(d.get("zeros", 0))
    return arr


def test_encode_matches_field_by_field():
    from spinoza_amd import _native as N
    from spinoza_amd.executor import encode_ops
    from spinoza_amd.workloads import hea, qft, random_circuit
    odd = [{"kind": 5, "target": np.int64(3), "theta": np.float32(1.5), "ones": 1 << 63},
           {"kind": np.int32(1), "classical": 1, "zeros": (1 << 70) + 5, "target": -1},
           {"kind": True, "theta": 2, "u": "0.25", "phi": np.float64(3)},
           {"kind": 4.0, "t1": 2 ** 33 + 7},
           types.MappingProxyType({"kind": 2, "target": 6}),
           collections.OrderedDict(kind=7, lam=0.5)]
    for ops in (odd, [], tuple(odd), random_circuit(7, 3, 1), qft(6), hea(5, 2, seed=2)[0]):
        arr, keep = encode_ops(ops)
        assert bytes(arr) == bytes(field_by_field(N, ops)) and keep == []
    assert bytes(encode_ops(collections.deque(odd))[0]) == bytes(encode_ops(odd)[0])


def test_encode_matrices_and_errors():
    from spinoza_amd import _native as N
    from spinoza_amd.executor import encode_ops
    u = np.array([[0, 1j], [1, 0]])
    arr, keep = encode_ops([{"kind": N.H}, {"kind": N.UNITARY, "target": 2, "matrix": u}])
    assert arr[1].m == 1 and arr[0].u_re is None and len(keep) == 2
    assert arr[1].u_re == keep[0].ctypes.data and arr[1].u_im == keep[1].ctypes.data
    assert np.array_equal(keep[0] + 1j * keep[1], u)
    for bad, err in (([{"target": 1}], KeyError), ([3], TypeError), ([{"kind": None}], TypeError),
                     ([{"kind": 1, "theta": "x"}], ValueError)):
        with pytest.raises(err):
            encode_ops(bad)
