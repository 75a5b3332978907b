"""Runs of a few ops on states of at most 12 qubits go op by op, longer ones in
one launch: amplitudes on either side of the line, in every mode."""
import numpy as np
import pytest

from test_plan_short import short_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 8, 12])
def test_short_runs_bit_identical(orc, n):
    import spinoza_amd as spz
    from spinoza_amd import _native as N
    from spinoza_amd.executor import run_ops
    base = orc.random_state(90 + n, n)
    for length in range(1, 9):
        print(f"case short n={n} length={length}", flush=True)
        ops = short_run(n, length, length)
        lengths = [length]
        if n > 1:  # a measurement between two runs, and a classical control
            lengths.append(1 + 9 - length)
            ops += [{"kind": N.M, "target": 0, "u": 0.3},
                    {"kind": N.X, "target": n - 1, "ones": 1, "classical": True}]
            ops += short_run(n, 9 - length, length + 20)
        for prec in ("f64", "f32"):
            p, *rest = (spz.State.from_arrays(base.re, base.im, prec) for _ in range(3))
            want = run_ops(p, ops, mode=N.EXEC_PLAIN)
            for s, mode in zip(rest, (N.EXEC_AUTO, N.EXEC_STRICT)):
                assert run_ops(s, ops, mode=mode) == want
                for x, y in zip(s.download(), p.download()):
                    if prec == "f64" or max(lengths) <= 5:  # (FP32: every run op by op)
                        assert np.array_equal(x, y), mode
                    else:  # PLAIN rounds after every gate, at most 2^-24 of an amplitude
                        assert np.max(np.abs(x - y)) < len(ops) * 2.0 ** -22
