"""Workloads that stand for what programs do with this framework.

Each listed case is one kind of use at one size; ``draw`` gives more of the
same kinds over their whole range.  A case is prepared once (the states,
encoded circuits and parameters a program keeps) and then run pass after pass
through the public entry points.  ``exact`` computes the same outputs in
complex128 with plain torch operations.

Paths:
  circuit   an encoded circuit on a state (executors AUTO, STRICT, DENSE5;
            FP64 or FP32 storage), with measurement samples where asked for
  gates     the functional gate calls, one after another
  mixed     a circuit with every arm of execute: dense blocks, swaps,
            mid-circuit measurement, classical control, bit-flip noise
  expect    x, y and z expectations of every qubit and the Ising energy
  grad      one optimiser step's forward and backward through torch.autograd
  batch     energies and gradients of many independent circuits in one call
"""
import math
import random

import numpy as np
import torch

import spinoza_amd as spz
from spinoza_amd import _native as N
from spinoza_amd.autograd import IsingEnergy, batch_adjoint
from spinoza_amd.executor import encode_ops, run_ops
from spinoza_amd.torch_interop import device_views

MODES = {"auto": N.EXEC_AUTO, "strict": N.EXEC_STRICT, "dense5": N.EXEC_DENSE5}
TWO_PI = 2.0 * math.pi


def listed():
    return [
        # the smallest calls: a teaching-size circuit run and sampled, where
        # launches and latency are everything
        {"name": "circuit_9q", "path": "circuit", "kind": "random", "n": 9, "layers": 6,
         "prec": "f64", "mode": "auto", "shots": 512},
        # an ordinary simulation of a mid-size circuit with measurement shots
        {"name": "circuit_17q", "path": "circuit", "kind": "random", "n": 17, "layers": 12,
         "prec": "f64", "mode": "auto", "shots": 1000},
        # the 20-qubit quantum Fourier transform of a loaded signal, 4096 shots
        {"name": "qft_20q", "path": "circuit", "kind": "qft", "n": 20, "layers": 1,
         "prec": "f64", "mode": "auto", "shots": 4096},
        # the headline workload: 1800 gates on a 16 GiB state
        {"name": "circuit_30q", "path": "circuit", "kind": "random", "n": 30, "layers": 40,
         "prec": "f64", "mode": "auto", "shots": 0},
        # the FP32 storage option, used to fit more qubits
        {"name": "circuit_f32_27q", "path": "circuit", "kind": "random", "n": 27, "layers": 15,
         "prec": "f32", "mode": "auto", "shots": 0},
        # the dense 5-qubit block executor
        {"name": "dense5_26q", "path": "circuit", "kind": "random", "n": 26, "layers": 6,
         "prec": "f64", "mode": "dense5", "shots": 0},
        # the functional API (gates::apply, c_apply, cc_apply), one pass per gate
        {"name": "gates_25q", "path": "gates", "n": 25, "count": 36, "prec": "f64"},
        # a circuit with measurement, classical control, noise and dense blocks
        {"name": "mixed_21q", "path": "mixed", "n": 21, "layers": 2, "blocks": 6, "measures": 7,
         "prec": "f64"},
        # observables of a prepared state
        {"name": "expect_23q", "path": "expect", "n": 23, "prec": "f64"},
        # a small variational step
        {"name": "grad_11q", "path": "grad", "n": 11, "layers": 4, "ckpt": 0, "prec": "f64"},
        # the large variational step: 480 parameters at 24 qubits
        {"name": "grad_24q", "path": "grad", "n": 24, "layers": 10, "ckpt": 142, "prec": "f64"},
        # a generation of independent small ansatz circuits, 10 to 18 qubits
        {"name": "batch_128", "path": "batch", "count": 128, "nmin": 10, "nmax": 18,
         "dmin": 2, "dmax": 12},
    ]


def draw(rng):
    """One more case of the same kinds: circuits from 4 to 29 qubits, gradients
    from 6 to 23, batches from a handful of circuits to about two hundred."""
    path = rng.choice(["circuit", "circuit", "circuit", "circuit", "gates", "mixed", "expect",
                       "grad", "grad", "batch"])
    prec = rng.choice(["f64", "f64", "f64", "f32"])
    if path == "circuit":
        mode = rng.choice(["auto", "auto", "auto", "strict", "dense5"])
        kind = rng.choice(["random", "random", "hea", "qft"]) if mode != "dense5" else "random"
        n = rng.randint(4, {"auto": 29, "strict": 27, "dense5": 26}[mode])
        layers = 1 if kind == "qft" else rng.randint(2, 5 if mode == "dense5" else 20)
        # (no shots from FP32 states: which index a uniform meets there hangs on
        # the last bits of the stored amplitudes)
        shots = rng.choice([0, 1, 100, 1000, 4096, 10000]) if n <= 26 and prec == "f64" else 0
        return {"path": path, "kind": kind, "n": n, "layers": layers, "prec": prec, "mode": mode,
                "shots": shots}
    if path == "gates":
        return {"path": path, "n": rng.randint(3, 27), "count": rng.randint(10, 50), "prec": prec}
    if path == "mixed":
        return {"path": path, "n": rng.randint(6, 24), "layers": rng.randint(1, 4),
                "blocks": rng.randint(1, 8), "measures": rng.randint(1, 6), "prec": prec}
    if path == "expect":
        return {"path": path, "n": rng.randint(4, 26), "prec": prec}
    if path == "grad":
        n = rng.randint(6, 23)
        return {"path": path, "n": n, "layers": rng.randint(1, 12),
                "ckpt": rng.choice([0, 0, 50, 97]), "prec": prec}
    nmin = rng.randint(4, 14)
    return {"path": path, "count": int(2.0 ** rng.uniform(2.0, 7.5)), "nmin": nmin,
            "nmax": rng.randint(nmin, 19), "dmin": rng.randint(1, 3), "dmax": rng.randint(4, 12)}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _op(kind, target, theta=0.0, phi=0.0, lam=0.0, **more):
    d = {"kind": kind, "target": target, "theta": theta, "phi": phi, "lam": lam, "t1": 0,
         "ones": 0, "zeros": 0, "classical": False}
    d.update(more)
    return d


def _random(n, layers, rng):
    """Per layer one gate of {H,X,Y,Z,RX,RY,RZ,P,U} on every qubit, then CX or
    CZ on a random matching."""
    ops = []
    for _ in range(layers):
        for q in range(n):
            kind = rng.choice([N.H, N.X, N.Y, N.Z, N.RX, N.RY, N.RZ, N.P, N.U])
            a = [rng.uniform(0.0, TWO_PI) for _ in range(3)]
            if kind == N.U:
                ops.append(_op(kind, q, *a))
            elif kind in (N.RX, N.RY, N.RZ, N.P):
                ops.append(_op(kind, q, a[0]))
            else:
                ops.append(_op(kind, q))
        perm = list(range(n))
        rng.shuffle(perm)
        for i in range(n // 2):
            ops.append(_op(rng.choice([N.X, N.Z]), perm[2 * i + 1], ones=1 << perm[2 * i]))
    return ops


def _hea(n, layers, thetas):
    """Per layer RY and RZ on every qubit, then a CX ladder; with the index of
    every parameter's op."""
    ops, where, k = [], [], 0
    for _ in range(layers):
        for q in range(n):
            where += [len(ops), len(ops) + 1]
            ops.append(_op(N.RY, q, thetas[k]))
            ops.append(_op(N.RZ, q, thetas[k + 1]))
            k += 2
        for q in range(n - 1):
            ops.append(_op(N.X, q + 1, ones=1 << q))
    return ops, where


def _qft(n):
    ops = []
    for j in range(n - 1, -1, -1):
        ops.append(_op(N.H, j))
        for k in range(j - 1, -1, -1):
            ops.append(_op(N.P, j, math.pi / float(2 ** (j - k)), ones=1 << k))
    for i in range(n // 2):
        ops.append(_op(N.SWAP, i, t1=n - 1 - i))
    return ops


def _unitary(m, rng):
    r = np.random.RandomState(rng.randrange(1 << 31))
    q, _ = np.linalg.qr(r.normal(size=(1 << m, 1 << m)) + 1j * r.normal(size=(1 << m, 1 << m)))
    return q


def _mixed(case, seed):
    n, rng = case["n"], random.Random(seed)
    ops = _random(n, case["layers"], rng)
    for _ in range(case["blocks"]):
        m = rng.randint(1, min(5, n - 1))
        t = rng.randint(0, n - m)
        out = [q for q in range(n) if not t <= q < t + m]
        ones = 1 << rng.choice(out) if rng.random() < 0.3 else 0
        ops.append(_op(N.UNITARY, t, matrix=_unitary(m, rng), ones=ones))
        a, b = rng.sample(range(n), 2)
        ops.append(_op(N.SWAP, a, t1=b))
        ops += _random(n, 1, rng)[: n // 2]
    for q in rng.sample(range(n), min(case["measures"], n - 2)):
        ops.append(_op(N.M, q, u=rng.random()))
        t = rng.choice([x for x in range(n) if x != q])
        ops.append(_op(N.RX, t, rng.uniform(0, TWO_PI), ones=1 << q, classical=True))
        ops.append(_op(N.BITFLIP, rng.randrange(n), 0.3, u=rng.random()))
        ops += _random(n, 1, rng)[: n // 3]
    return ops


def _calls(case, seed):
    """(gate kind, three angles, controls, target or two swapped qubits)."""
    n, rng, out = case["n"], random.Random(seed), []
    for i in range(case["count"]):
        kind = rng.choice([N.H, N.X, N.Y, N.Z, N.RX, N.RY, N.RZ, N.P, N.U, N.SWAP])
        a = [rng.uniform(0.0, TWO_PI) for _ in range(3)]
        nc = 0 if kind == N.SWAP else rng.choice([0, 0, 0, 1, 1, 2])
        qs = rng.sample(range(n), 2 if kind == N.SWAP else 1 + min(nc, n - 1))
        out.append((kind, a, qs[1:], qs[0]))
    return out


def _circuit(case, seed):
    rng = random.Random(seed)
    if case["kind"] == "qft":
        return _qft(case["n"])
    if case["kind"] == "hea":
        th = [rng.uniform(0.0, TWO_PI) for _ in range(2 * case["n"] * case["layers"])]
        return _hea(case["n"], case["layers"], th)[0]
    return _random(case["n"], case["layers"], rng)


def _batch(case, seed):
    # the circuits' shapes belong to the case, their angles to the seed
    shapes, rng, out = random.Random(case["count"]), random.Random(seed), []
    for _ in range(case["count"]):
        n = shapes.randint(case["nmin"], case["nmax"])
        depth = shapes.randint(case["dmin"], case["dmax"])
        out.append((n, _hea(n, depth, [rng.uniform(0.0, TWO_PI) for _ in range(2 * n * depth)])[0]))
    return out


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _gaussian(n, seed):
    """A normalised state with independent normal parts."""
    g = torch.Generator(device=_device()).manual_seed(seed)
    re = torch.randn(1 << n, generator=g, dtype=torch.float64, device=_device())
    im = torch.randn(1 << n, generator=g, dtype=torch.float64, device=_device())
    s = 1.0 / torch.sqrt(re.square().sum() + im.square().sum())
    return re * s, im * s


def _views(state):
    """The state's amplitudes as tensors that keep the state alive."""
    views = device_views(state)
    for v in views:
        v.owner = state
    return views


def _loaded(case, seed):
    s = spz.State(case["n"], case["prec"])
    for v, x in zip(device_views(s), _gaussian(case["n"], seed)):
        v.copy_(x)
    return s


def _uniforms(case, seed):
    return np.random.RandomState(seed % (1 << 31)).random_sample(case["shots"])


def prepare(case, seed):
    path = case["path"]
    if path == "batch":
        return {"case": case, "circuits": _batch(case, seed)}
    n, prec = case["n"], case.get("prec", "f64")
    st = {"case": case}
    if path == "grad":
        rng = random.Random(seed)
        th = [rng.uniform(0.0, TWO_PI) for _ in range(2 * n * case["layers"])]
        st["thetas"] = torch.tensor(th, dtype=torch.float64, device=_device(), requires_grad=True)
        st["build"] = lambda vals: _hea(n, case["layers"], vals)
        return st
    if path in ("gates", "expect"):
        st["state"] = _loaded(case, seed)
    else:
        st["state"] = spz.State(n, prec)
        st["ops"] = _circuit(case, seed) if path == "circuit" else _mixed(case, seed)
        st["encoded"] = encode_ops(st["ops"])
        st["source"] = _loaded(case, seed) if case.get("kind") == "qft" else None
        if case.get("shots"):
            st["uniforms"] = _uniforms(case, seed)
    if path == "gates":
        st["calls"] = [(spz.Gate(k, *a) if k != N.SWAP else spz.Gate.SWAP(t, c[0]), c, t)
                       for k, a, c, t in _calls(case, seed)]
    st["views"] = _views(st["state"])
    return st


def run(st):
    case = st["case"]
    path = case["path"]
    if path == "batch":
        energies, grads, _ = batch_adjoint(st["circuits"], 1.0, wg_max_qubits=18)
        return {"energies": energies, "grads": np.concatenate(grads)}
    if path == "grad":
        th = st["thetas"]
        th.grad = None
        e = IsingEnergy.apply(th, st["build"], case["n"], 1.0, case["ckpt"], case["prec"])
        e.backward()
        return {"energy": e.detach(), "grad": th.grad}
    s = st["state"]
    if path == "expect":
        targets = list(range(case["n"]))
        out = {o: np.array(spz.xyz_expectation_value(o, s, targets)) for o in "xyz"}
        out["energy"] = np.float64(spz.ising_energy(s, 1.0))
        return out
    if path == "gates":
        for gate, controls, target in st["calls"]:
            if gate.kind == N.SWAP or not controls:
                spz.apply(gate, s, target)
            elif len(controls) == 1:
                spz.c_apply(gate, s, controls[0], target)
            else:
                spz.cc_apply(gate, s, controls[0], controls[1], target)
        return st["views"]
    # circuits start from |0...0>, or from the loaded signal
    if st["source"] is None:
        s.set_basis(0)
    else:
        s.copy_from(st["source"])
    if path == "mixed":
        outcomes = run_ops(s, st["ops"], encoded=st["encoded"])
        return {"state": st["views"], "outcomes": np.array(outcomes)}
    run_ops(s, st["ops"], mode=MODES[case["mode"]], encoded=st["encoded"])
    if not case["shots"]:
        return {"state": st["views"]}
    shots = spz.sample(s, st["uniforms"])
    return {"state": st["views"], "shots": shots.astype(np.int64)}


# ---------------------------------------------------------------------------
# The work of one pass
# ---------------------------------------------------------------------------
# real operations per amplitude of an uncontrolled gate (products and sums)
_FLOPS = {N.H: 4, N.X: 0, N.Y: 0, N.Z: 0.5, N.P: 3, N.RX: 6, N.RY: 6, N.RZ: 6, N.U: 14,
          N.SWAP: 0, N.BITFLIP: 0, N.M: 3}


def _flops(ops, n):
    total = 0.0
    for o in ops:
        per = 8.0 * len(o["matrix"]) if "matrix" in o else _FLOPS[o["kind"]]
        total += per * 2.0 ** (n - bin(o["ones"] | o["zeros"]).count("1"))
    return total


def work(case):
    path = case["path"]
    amp = 8.0 if case.get("prec") == "f32" else 16.0
    if path == "batch":
        circuits = _batch(case, 1)
        return {"bytes": sum(8.0 * len(ops) for _, ops in circuits),
                "flops": sum(3.0 * _flops(ops, n) for n, ops in circuits)}
    n = case["n"]
    size = amp * 2.0 ** n
    if path == "grad":
        ops, where = _hea(n, case["layers"], [0.0] * (2 * n * case["layers"]))
        # forward, and the reverse sweep of the state and of its dual; the
        # gradients' inner products
        return {"bytes": 8.0 * len(where),
                "flops": 3.0 * _flops(ops, n) + 8.0 * len(where) * 2.0 ** n}
    if path == "expect":
        return {"bytes": size, "flops": 2.0 ** n * (3 * 4.0 * n + 3.0 * n)}
    if path == "gates":
        flops = 0.0
        for k, _, c, _t in _calls(case, 1):
            flops += _FLOPS[k] * 2.0 ** (n - (0 if k == N.SWAP else len(c)))
        return {"bytes": 2.0 * size, "flops": flops}
    if path == "mixed":
        return {"bytes": size, "flops": _flops(_mixed(case, 1), n)}
    # the circuit's result is written once; a loaded signal is read once
    return {"bytes": size * (2.0 if case["kind"] == "qft" else 1.0),
            "flops": _flops(_circuit(case, 1), n)}


# ---------------------------------------------------------------------------
# The same outputs in complex128
# ---------------------------------------------------------------------------
def _matrix(kind, th, ph, la):
    c, s = math.cos(th / 2), math.sin(th / 2)
    h = math.sqrt(0.5)
    e = lambda x: complex(math.cos(x), math.sin(x))  # noqa: E731
    return {N.H: [[h, h], [h, -h]], N.X: [[0, 1], [1, 0]], N.Y: [[0, -1j], [1j, 0]],
            N.Z: [[1, 0], [0, -1]], N.P: [[1, 0], [0, e(th)]],
            N.RX: [[c, -1j * s], [-1j * s, c]], N.RY: [[c, -s], [s, c]],
            N.RZ: [[e(-th / 2), 0], [0, e(th / 2)]],
            N.U: [[c, -e(la) * s], [e(ph) * s, e(ph + la) * c]]}[kind]


def _halves(psi, n, target, controls):
    """psi's amplitudes whose controls read 1, split by the target bit, as views."""
    v = psi.view([2] * n) if n else psi
    at = [slice(None)] * n
    for c in controls:
        at[n - 1 - c] = 1
    lo, hi = list(at), list(at)
    lo[n - 1 - target], hi[n - 1 - target] = 0, 1
    return v[tuple(lo)], v[tuple(hi)]


def _bits(mask):
    return [q for q in range(64) if (mask >> q) & 1]


def _gate(psi, n, m, target, controls):
    a, b = _halves(psi, n, target, controls)
    if m[0][1] == 0 and m[1][0] == 0:
        if m[0][0] != 1:
            a *= m[0][0]
        if m[1][1] != 1:
            b *= m[1][1]
        return
    x = a * m[0][0] + b * m[0][1]
    b.copy_(a * m[1][0] + b * m[1][1])
    a.copy_(x)


def _swap(psi, n, p, q):
    v = psi.view([2] * n)
    at, bt = [slice(None)] * n, [slice(None)] * n
    at[n - 1 - p], at[n - 1 - q], bt[n - 1 - p], bt[n - 1 - q] = 0, 1, 1, 0
    x = v[tuple(at)].clone()
    v[tuple(at)] = v[tuple(bt)]
    v[tuple(bt)] = x


def _dense(psi, n, mat, t, controls):
    m = len(mat).bit_length() - 1
    u = torch.tensor(mat, dtype=torch.complex128, device=psi.device)
    v = psi.view(-1, 1 << m, 1 << t)
    out = torch.zeros_like(v)
    for r in range(1 << m):
        for c in range(1 << m):
            out[:, r] += u[r, c] * v[:, c]
    if controls:  # the rest stays as it was
        c = controls[0]
        keep = psi.view(-1, 2, 1 << c)[:, 0].clone()
        psi.copy_(out.view(-1))
        psi.view(-1, 2, 1 << c)[:, 0] = keep
    else:
        psi.copy_(out.view(-1))


def _simulate(psi, n, ops):
    """Runs ops on psi in place; the outcome of each (255: none)."""
    outcomes, seen = [], {}
    for o in ops:
        out, kind, controls = 255, o["kind"], _bits(o["ones"])
        if kind == N.M:
            if o["target"] not in seen:
                a, b = _halves(psi, n, o["target"], [])
                p0 = float(a.abs().square().sum())
                out = 1 if o["u"] < 1.0 - p0 else 0
                keep = (b if out else a) / math.sqrt(1.0 - p0 if out else p0)
                a.copy_(keep)  # the measured qubit is reset to |0>
                b.zero_()
                seen[o["target"]] = out
        elif kind == N.BITFLIP:
            if o["u"] <= o["theta"]:
                _gate(psi, n, [[0, 1], [1, 0]], o["target"], [])
        elif kind == N.SWAP:
            _swap(psi, n, o["target"], o["t1"])
        elif kind == N.UNITARY:
            _dense(psi, n, o["matrix"], o["target"], controls)
        else:
            m = _matrix(kind, o["theta"], o["phi"], o["lam"])
            if o["classical"] and controls[0] in seen:
                if seen[controls[0]]:
                    _gate(psi, n, m, o["target"], [])
            else:
                _gate(psi, n, m, o["target"], controls)
        outcomes.append(out)
    return outcomes


def _zero(n):
    psi = torch.zeros(1 << n, dtype=torch.complex128, device=_device())
    psi[0] = 1.0
    return psi


def _split(psi, prec):
    del prec  # the exact values, not what the storage type can hold
    return [psi.real.clone(), psi.imag.clone()]


def _parity(n, q, dev):
    return 1.0 - 2.0 * ((torch.arange(1 << n, device=dev) >> q) & 1).double()


def _ising(psi, n):
    """H psi for H = sum Z_i Z_{i+1} + sum X_i."""
    diag = torch.zeros(1 << n, dtype=torch.float64, device=psi.device)
    z = _parity(n, 0, psi.device)
    for i in range(n - 1):
        w = _parity(n, i + 1, psi.device)
        diag += z * w
        z = w
    out = diag * psi
    for i in range(n):
        out.view(-1, 2, 1 << i).add_(psi.view(-1, 2, 1 << i).flip(1))
    return out


def _dot(a, b):
    return torch.sum(a.conj() * b)


def _adjoint(n, ops):
    """Energy and dE/dtheta of every RY and RZ (zero for the others)."""
    psi = _zero(n)
    _simulate(psi, n, ops)
    lam = _ising(psi, n)
    energy = _dot(psi, lam).real
    grads = [None] * len(ops)
    for k in range(len(ops) - 1, -1, -1):
        o = ops[k]
        c = _bits(o["ones"])
        a, b = _halves(psi, n, o["target"], c)
        la, lb = _halves(lam, n, o["target"], c)
        if o["kind"] == N.RY:  # Im <lam|Y|psi>
            grads[k] = (_dot(la, -1j * b) + _dot(lb, 1j * a)).imag
        elif o["kind"] == N.RZ:
            grads[k] = (_dot(la, a) - _dot(lb, b)).imag
        m = _matrix(o["kind"], -o["theta"], o["phi"], o["lam"])
        _gate(psi, n, m, o["target"], c)
        _gate(lam, n, m, o["target"], c)
    zero = torch.zeros((), dtype=torch.float64, device=psi.device)
    return energy, torch.stack([zero if g is None else g for g in grads])


def exact(case, seed):
    path = case["path"]
    if path == "batch":
        if sum(len(ops) for _, ops in _batch(case, 1)) > 40000:
            return None
        got = [_adjoint(n, ops) for n, ops in _batch(case, seed)]
        return {"energies": torch.stack([e for e, _ in got]),
                "grads": torch.cat([g for _, g in got])}
    n = case["n"]
    if path == "grad":
        rng = random.Random(seed)
        th = [rng.uniform(0.0, TWO_PI) for _ in range(2 * n * case["layers"])]
        ops, where = _hea(n, case["layers"], th)
        e, g = _adjoint(n, ops)
        return {"energy": e, "grad": g[where]}
    if path in ("expect", "gates"):
        re, im = _gaussian(n, seed)
        if case["prec"] == "f32":
            re, im = re.float().double(), im.float().double()
        psi = torch.complex(re, im)
    if path == "expect":
        out = {"x": [], "y": [], "z": []}
        for q in range(n):
            a, b = _halves(psi, n, q, [])
            ab = _dot(a, b)
            out["x"].append(2.0 * float(ab.real))
            out["y"].append(2.0 * float(ab.imag))
            out["z"].append(float(a.abs().square().sum() - b.abs().square().sum()))
        out = {k: torch.tensor(v, dtype=torch.float64) for k, v in out.items()}
        out["energy"] = _dot(psi, _ising(psi, n)).real
        return out
    if path == "gates":
        for k, a, c, t in _calls(case, seed):
            if k == N.SWAP:
                _swap(psi, n, t, c[0])
            else:
                _gate(psi, n, _matrix(k, *a), t, c)
        return tuple(_split(psi, case["prec"]))
    ops = _circuit(case, seed) if path == "circuit" else _mixed(case, seed)
    if len(ops) * 2.0 ** n > 1000 * 2.0 ** 28:
        return None  # minutes in complex128
    if case.get("kind") == "qft":
        re, im = _gaussian(n, seed)
        if case["prec"] == "f32":
            re, im = re.float().double(), im.float().double()
        psi = torch.complex(re, im)
    else:
        psi = _zero(n)
    _simulate(psi, n, ops)
    return {"state": _split(psi, case["prec"])}
