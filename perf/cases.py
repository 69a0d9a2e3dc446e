"""Timed work of the state-vector engine: what programs that use it spend their time on.

Kinds of case, each through the public entry points a program calls:

  gates    one brick layer (H, R{X,Y,Z}, CNOT ladder) gate by gate through QubitRegister --
           the plain way to run a circuit, from a few qubits (call latency) to 30
  qft      quantum Fourier transform, gate by gate: Hadamards, controlled phases, swaps
  fused    the same kind of circuits with TurnOnFusion: brick layers, or random dense 1- and
           2-qubit gates
  qaoa     MaxCut QAOA: cost and the adjoint gradient of every angle (forward and backward),
           unit and weighted graphs
  hea      a batch of hardware-efficient-ansatz circuits: costs and all gradients
  readout  reordering the qubits (PermuteQubits), then the terms of an Ising energy, a few
           longer Pauli strings, the norm and an overlap
  pool     a pool of noisy trajectories: common gates, per-state noise gates, per-state readout

`prepare` makes what a program holds before the call (registers with a generic state, gate
lists, angles) from the seed; `run` is one pass; `work` what a pass cannot do without;
`exact` the same result in 64 bits with plain torch.
"""
import math
import os
import random
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.abspath(os.getcwd()), "intel-qs_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

ROTATIONS = ("ApplyRotationX", "ApplyRotationY", "ApplyRotationZ")


# ---------------------------------------------------------------------------------------
# Cases


def listed():
    return [
        # A small circuit gate by gate: nothing but the cost of a call and a launch.
        dict(name="gates_10q_dp", kind="gates", n=10, dp=True, layers=1),
        # The size a workstation CPU still runs; the state lives in the GPU's caches.
        dict(name="gates_20q_dp", kind="gates", n=20, dp=True, layers=2),
        # The headline circuit: 30 qubits, every gate a pass over 16 GiB.
        dict(name="gates_30q_dp", kind="gates", n=30, dp=True, layers=1),
        # A textbook algorithm at an odd size in single precision: 325 gates.
        dict(name="qft_25q_sp", kind="qft", n=25, dp=False, reach=24),
        # Fusion on a cache-sized register, where host planning and launches count.
        dict(name="fused_brick_20q_dp", kind="fused", n=20, dp=True, gates="brick", count=10),
        # Fusion on a large register: random dense gates, no structure to use.
        dict(name="fused_random_30q_sp", kind="fused", n=30, dp=False, gates="random", count=120),
        # A QAOA optimizer's inner step on a small graph (latency of many short passes).
        dict(name="qaoa_14q_dp", kind="qaoa", n=14, dp=True, p=6, weighted=False),
        # The same on the largest graph of the gradient benchmark.
        dict(name="qaoa_28q_dp", kind="qaoa", n=28, dp=True, p=8, weighted=False),
        # Weighted graph, odd size, single precision.
        dict(name="qaoa_25q_sp_weighted", kind="qaoa", n=25, dp=False, p=4, weighted=True),
        # One optimizer step for a batch of ansatz circuits of mixed size.
        dict(name="hea_64x10_22q_sp", kind="hea", count=64, qmin=10, qmax=22, dmin=10, dmax=50, dp=False, pick=6),
        # Energy readout of a finished state after bringing its qubits into another order.
        dict(name="readout_27q_dp", kind="readout", n=27, dp=True, bonds=26),
        # Noisy trajectories of a small device, all states in one register.
        dict(name="pool_32x16q_dp", kind="pool", n=16, states=32, layers=2),
    ]


def draw(rng):
    kind = rng.choice(("gates", "gates", "qft", "fused", "fused", "qaoa", "qaoa", "hea", "readout", "pool"))
    dp = rng.random() < 0.5
    if kind == "gates":
        n = rng.randint(8, 30)
        return dict(kind=kind, n=n, dp=dp, layers=1 if n > 27 else rng.randint(1, 7 if n < 26 else 4))
    if kind == "qft":
        n = rng.randint(8, 27)
        return dict(kind=kind, n=n, dp=dp, reach=rng.randint(4, n - 1))
    if kind == "fused":
        gates = rng.choice(("brick", "random"))
        n = rng.randint(9, 30)
        if gates == "brick":
            return dict(kind=kind, n=n, dp=dp, gates=gates, count=rng.randint(1, 3 if n > 27 else 12))
        return dict(kind=kind, n=n, dp=dp, gates=gates, count=rng.randint(10, 100 if n > 27 else 200))
    if kind == "qaoa":
        n = rng.randint(10, 28)
        return dict(kind=kind, n=n, dp=dp, p=rng.randint(1, 8), weighted=rng.random() < 0.3)
    if kind == "hea":
        qmin = rng.randint(4, 12)
        return dict(kind=kind, count=int(round(2 ** rng.uniform(2, 6))), qmin=qmin, qmax=rng.randint(qmin, 22),
                    dmin=2, dmax=rng.randint(4, 50), dp=dp, pick=rng.randint(0, 1 << 20))
    if kind == "readout":
        n = rng.randint(9, 29)
        return dict(kind=kind, n=n, dp=dp, bonds=rng.randint(n // 2, 2 * n))
    n = rng.randint(6, 20)
    return dict(kind="pool", n=n, states=int(round(2 ** rng.uniform(1, min(6.0, 26.0 - n)))), layers=rng.randint(1, 3))


# ---------------------------------------------------------------------------------------
# Inputs


def _f32(x):
    """An angle that single and double precision hold alike."""
    return float(np.float32(x))


def _amplitudes(case, seed):
    """A generic normalized state (complex Gaussian), as after a deep circuit."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    real = torch.float64 if case["dp"] else torch.float32
    a = torch.randn(1 << case["n"], 2, generator=g, device="cuda", dtype=real)
    return torch.view_as_complex(a.mul_(1.0 / float(torch.linalg.vector_norm(a, dtype=torch.float64))))


def _brick(n, layers, rng):
    ops = []
    for layer in range(layers):
        ops += [("ApplyHadamard", q) for q in range(n)]
        ops += [(rng.choice(ROTATIONS), q, _f32(rng.uniform(0.0, 2.0 * math.pi))) for q in range(n)]
        ops += [("ApplyCPauliX", q, q + 1) for q in range(layer % 2, n - 1, 2)]
    return ops


def _unitary(d, rng, dtype):
    z = rng.standard_normal((d, d)) + 1j * rng.standard_normal((d, d))
    q, r = np.linalg.qr(z)
    return np.ascontiguousarray((q * (np.diag(r) / np.abs(np.diag(r)))).astype(dtype))


def _random_gates(n, count, seed, dtype):
    rng = np.random.default_rng(seed)
    ops = []
    for _ in range(count):
        if rng.random() < 0.5:
            ops.append(("Apply1QubitGate", int(rng.integers(n)), _unitary(2, rng, dtype)))
        else:
            a, b = (int(x) for x in rng.choice(n, 2, replace=False))
            ops.append(("Apply2QubitGate", a, b, _unitary(4, rng, dtype)))
    return ops


def _qft(n, reach):
    """High qubit first, each Hadamard followed by its controlled phases (from qubits at most
    `reach` away: n - 1 for the full transform, less for the approximate one), then the swaps
    that reverse the qubit order."""
    ops = []
    for t in range(n - 1, -1, -1):
        ops.append(("ApplyHadamard", t))
        ops += [("ApplyCPhaseRotation", c, t, _f32(math.pi / (1 << (t - c)))) for c in range(t - 1, max(t - reach, 0) - 1, -1)]
    return ops + [("ApplySwap", q, n - 1 - q) for q in range(n // 2)]


def _ops(case, seed):
    n = case["n"]
    if case["kind"] == "qft":
        return _qft(n, case["reach"])
    if case["kind"] == "gates":
        return _brick(n, case["layers"], random.Random(seed))
    if case["gates"] == "brick":
        return _brick(n, case["count"], random.Random(seed))
    return _random_gates(n, case["count"], seed, np.complex128 if case["dp"] else np.complex64)


def _graph(case, seed):
    """A random graph of about 1.5 edges per vertex."""
    n, rng = case["n"], random.Random(seed)
    pairs = [(u, v) for u in range(n) for v in range(u + 1, n)]
    edges = sorted(rng.sample(pairs, (3 * n) // 2))
    return [(u, v, _f32(rng.uniform(0.25, 2.0)) if case["weighted"] else 1.0) for u, v in edges]


def _angles(case, seed):
    rng = random.Random(seed + 1)
    return [[rng.uniform(0.0, math.pi) for _ in range(case["p"])] for _ in range(2)]


def _hea_sizes(case):
    """Sizes of the batch's circuits (part of the case), the largest of its range among them."""
    rng = random.Random(case["pick"])
    nq = [rng.randint(case["qmin"], case["qmax"]) for _ in range(case["count"])]
    nq[0] = case["qmax"]
    return nq, [rng.randint(case["dmin"], case["dmax"]) for _ in range(case["count"])]


def _hea_angles(case, seed):
    nq, dp = _hea_sizes(case)
    return np.random.default_rng(seed).uniform(0.0, 2.0 * math.pi, 2 * sum(a * b for a, b in zip(nq, dp)))


def _correlators(n):
    """Pauli strings (qubits, observables with X, Y, Z = 1, 2, 3) that a program reads besides
    the energy terms."""
    last, mid = n - 1, n // 2
    return [([0, last], [1, 1]), ([0, mid, last], [1, 2, 3]), ([1, mid], [2, 2]), ([0, 1, mid, last], [3, 1, 1, 3])]


def _bonds(case):
    """The coupled qubits of the energy: a chain, then random pairs."""
    n, rng = case["n"], random.Random(case["bonds"])
    pairs = [(q, q + 1) for q in range(n - 1)][:case["bonds"]]
    return pairs + [tuple(rng.sample(range(n), 2)) for _ in range(case["bonds"] - len(pairs))]


def _order(n, seed):
    order = list(range(n))
    random.Random(seed).shuffle(order)
    return order


class _Amplitudes:
    """A register's device memory for torch; the register lives as long as a tensor on it."""

    def __init__(self, register, pointer, n, dp):
        self.register = register
        self.__cuda_array_interface__ = dict(shape=(1 << n,), typestr="<c16" if dp else "<c8",
                                             data=(int(pointer), False), version=2, strides=None)


def _view(reg, n, dp):
    import ctypes

    from iqs_amd._lib import call

    p = ctypes.c_void_p()
    call("iqsh_info", ctypes.c_void_p(reg.DeviceHandle()), None, None, ctypes.byref(p))
    return torch.as_tensor(_Amplitudes(reg, p.value, n, dp), device="cuda")


def _register(case, seed):
    """A QubitRegister that holds the state of `_amplitudes`."""
    import intelqs_py as iqs
    from iqs_amd._lib import lib

    lib()
    n, dp = case["n"], case["dp"]
    reg = (iqs.QubitRegister if dp else iqs.QubitRegisterSP)(n, "base", 0, 0)
    state = _view(reg, n, dp)
    state.copy_(_amplitudes(case, seed))
    return reg, state


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("gates", "qft", "fused"):
        reg, state = _register(case, seed)
        calls = [(getattr(reg, op[0]), op[1:]) for op in _ops(case, seed)]
        return dict(kind=kind, reg=reg, state=state, calls=calls)
    if kind == "qaoa":
        from iqs_amd.qaoa import MaxCutQaoa

        gammas, betas = _angles(case, seed)
        problem = MaxCutQaoa(case["n"], _graph(case, seed), "c128" if case["dp"] else "c64")
        return dict(kind=kind, problem=problem, gammas=gammas, betas=betas, dp=case["dp"])
    if kind == "hea":
        from iqs_amd.batch import HeaBatch

        nq, dp = _hea_sizes(case)
        batch = HeaBatch(nq, dp, "c128" if case["dp"] else "c64")
        return dict(kind=kind, batch=batch, angles=_hea_angles(case, seed), dp=case["dp"])
    if kind == "readout":
        reg, _ = _register(case, seed)
        other, _ = _register(case, seed + 1000003)
        orders = [_order(case["n"], seed), list(range(case["n"]))]
        return dict(kind=kind, case=case, reg=reg, other=other, orders=orders, bonds=_bonds(case), turn=0)
    import intelqs_py as iqs
    from iqs_amd._lib import lib

    lib()
    pool = iqs.StatePool(case["n"], case["states"], "++++", 0)
    pool.SetSeedStreamPtrs(1 + seed % (1 << 30))
    pool.SetNoiseTimescales(60.0, 40.0)
    reg = pool.Register()
    layers = [[(getattr(reg, op[0]), op[1:]) for op in _brick(case["n"], 1, random.Random(seed + k))]
              for k in range(case["layers"])]
    return dict(kind=kind, pool=pool, layers=layers, n=case["n"], state=_view(reg, reg.NumQubits(), True))


# ---------------------------------------------------------------------------------------
# One pass


def run(state):
    kind = state["kind"]
    if kind in ("gates", "qft"):
        for gate, args in state["calls"]:
            gate(*args)
        return state["state"]
    if kind == "fused":
        reg = state["reg"]
        reg.TurnOnFusion()
        for gate, args in state["calls"]:
            gate(*args)
        reg.TurnOffFusion()
        return state["state"]
    if kind == "qaoa":
        cost, dgammas, dbetas = state["problem"].adjoint(state["gammas"], state["betas"])
        return _values(state["dp"], cost=[cost], gammas=dgammas, betas=dbetas)
    if kind == "hea":
        cost, grad = state["batch"].evaluate(state["angles"], grad=True)
        return _values(state["dp"], cost=cost, grad=grad)
    if kind == "readout":
        return _readout(state)
    pool = state["pool"]
    for layer in state["layers"]:
        for gate, args in layer:
            gate(*args)
        for q in range(state["n"]):
            pool.ApplyNoiseGate(q, 1.0)
    return dict(prob=np.array([pool.GetProbability(q) for q in range(state["n"])]), norm=np.array(pool.ComputeNorm()),
                zz=np.array([pool.ExpectationValueZString([q, q + 1]) for q in range(state["n"] - 1)]),
                state=state["state"])


def _values(dp, **values):
    """Read values in the precision of the amplitudes that they were taken from."""
    return {k: np.asarray(v, dtype=np.float64 if dp else np.float32) for k, v in values.items()}


def _readout(state):
    case, reg, other = state["case"], state["reg"], state["other"]
    n = case["n"]
    order = state["orders"][state["turn"]]  # there and back, pass by pass
    state["turn"] ^= 1
    reg.PermuteQubits(order, "direct")
    other.PermuteQubits(order, "direct")
    x = [reg.ExpectationValueX(q) for q in range(n)]
    z = [reg.GetProbability(q) for q in range(n)]
    zz = [reg.ExpectationValue([a, b], [3, 3], 1.0) for a, b in state["bonds"]]
    strings = [reg.ExpectationValue(list(q), list(o), 1.0) for q, o in _correlators(n)]
    overlap = reg.ComputeOverlap(other)
    return dict(_values(case["dp"], x=x, z=z, zz=zz, strings=strings, norm=[reg.ComputeNorm()],
                        overlap=[overlap.real, overlap.imag]), state=_view(reg, n, case["dp"]))


# ---------------------------------------------------------------------------------------
# What a pass cannot do without


def _gate_work(op, size, esz):
    """(bytes, flops) of one gate call on `size` amplitudes: the amplitudes it changes, read and
    written once; products with ones and zeros are none."""
    name = op[0]
    if name == "ApplyCPauliX" or name == "ApplySwap":
        return size * esz, 0
    if name == "ApplyCPhaseRotation":
        return size * esz // 2, size // 4 * 6
    if name == "ApplyRotationZ":
        return 2 * size * esz, size * 6
    if name == "Apply2QubitGate":
        return 2 * size * esz, size * 30
    if name == "Apply1QubitGate":
        return 2 * size * esz, size * 14
    return 2 * size * esz, size * 6  # real, or real and imaginary, 2x2 matrices


def work(case):
    kind = case["kind"]
    if kind == "hea":
        # Registers up to 12 qubits or so stay on the chip; each pair of angles is two products
        # per amplitude forward, and the undoing of both states and two inner products backward.
        flops = sum(d * (26 * n + 18) * (1 << n) for n, d in zip(*_hea_sizes(case)))
        return dict(bytes=2 * 8 * len(_hea_angles(case, 0)), flops=flops)
    if kind == "pool":
        size, esz = case["states"] << case["n"], 16
        gates = [_gate_work(op, size, esz) for op in _brick(case["n"], case["layers"], random.Random(0))]
        nbytes = sum(b for b, _ in gates) + case["layers"] * case["n"] * 2 * size * esz
        nbytes += case["n"] * size * esz // 2 + case["n"] * size * esz
        return dict(bytes=nbytes, flops=sum(f for _, f in gates) + case["layers"] * case["n"] * 14 * size)
    size, esz = 1 << case["n"], 16 if case["dp"] else 8
    if kind in ("gates", "qft"):
        gates = [_gate_work(op, size, esz) for op in _ops(case, 0)]
        return dict(bytes=sum(b for b, _ in gates), flops=sum(f for _, f in gates))
    if kind == "fused":
        return dict(bytes=2 * size * esz, flops=sum(_gate_work(op, size, esz)[1] for op in _ops(case, 0)))
    if kind == "qaoa":
        # A layer mixes every amplitude with every other, so the state passes once per layer
        # forward and, with lambda, once per layer backward.
        n, p = case["n"], case["p"]
        return dict(bytes=(2 * p + 4 * p + 2) * size * esz, flops=p * size * (6 * n + 6 + 16 * n + 18))
    n = case["n"]
    return dict(bytes=(4 + n + case["bonds"] + 4 + 1 + 2) * size * esz + n * size * esz // 2,
                flops=size * 6 * (2 * n + case["bonds"] + 7))


# ---------------------------------------------------------------------------------------
# The same in 64 bits with plain torch

_R = 1.0 / math.sqrt(2.0)


def _matrix(op):
    name, a = op[0], op[-1]
    if name == "ApplyHadamard":
        return np.array([[_R, _R], [_R, -_R]], dtype=np.complex128)
    if name == "ApplyRotationX":
        return np.array([[math.cos(a / 2), -1j * math.sin(a / 2)], [-1j * math.sin(a / 2), math.cos(a / 2)]])
    if name == "ApplyRotationY":
        return np.array([[math.cos(a / 2), -math.sin(a / 2)], [math.sin(a / 2), math.cos(a / 2)]], dtype=np.complex128)
    if name == "ApplyRotationZ":
        return np.diag([np.exp(-0.5j * a), np.exp(0.5j * a)])
    return np.asarray(a, dtype=np.complex128)


def _pairs(psi, q):
    v = psi.view(-1, 2, 1 << q)
    return v[:, 0], v[:, 1]


def _quads(psi, a, b):
    """The four parts of psi by (bit a, bit b)."""
    hi, lo = max(a, b), min(a, b)
    v = psi.view(-1, 2, 1 << (hi - lo - 1), 2, 1 << lo)
    return [[v[:, i, :, j] if a == hi else v[:, j, :, i] for j in (0, 1)] for i in (0, 1)]


def _mix(m, parts):
    new = []
    for row in m:
        acc = None
        for c, part in zip(row, parts):
            if c != 0:
                acc = part * complex(c) if acc is None else acc.add_(part * complex(c))
        new.append(acc)
    for part, x in zip(parts, new):
        part.copy_(x)


def _apply(psi, op):
    name = op[0]
    if name == "ApplyCPauliX":
        x, y = _quads(psi, op[1], op[2])[1]
        t = x.clone()
        x.copy_(y)
        y.copy_(t)
    elif name == "ApplySwap":
        q = _quads(psi, op[1], op[2])
        t = q[0][1].clone()
        q[0][1].copy_(q[1][0])
        q[1][0].copy_(t)
    elif name == "ApplyCPhaseRotation":
        _quads(psi, op[1], op[2])[1][1].mul_(complex(math.cos(op[3]), math.sin(op[3])))
    elif name == "Apply2QubitGate":
        q = _quads(psi, op[1], op[2])
        _mix(_matrix(op), [q[0][0], q[0][1], q[1][0], q[1][1]])
    else:
        _mix(_matrix(op), list(_pairs(psi, op[1])))


def _im(lam, psi):
    """Im sum conj(lam) psi."""
    return float((lam.real * psi.imag).sum() - (lam.imag * psi.real).sum())


def _exact_qaoa(case, seed):
    n, edges = case["n"], _graph(case, seed)
    gammas, betas = _angles(case, seed)
    cut = torch.zeros(1 << n, dtype=torch.float64, device="cuda")
    for u, v, w in edges:
        q = _quads(cut, u, v)
        q[0][1].add_(w)
        q[1][0].add_(w)
    psi = torch.full((1 << n,), 1.0 / math.sqrt(float(1 << n)), dtype=torch.complex128, device="cuda")
    for g, b in zip(gammas, betas):
        psi.mul_(torch.polar(torch.ones_like(cut), -g * cut))
        for q in range(n):
            _apply(psi, ("ApplyRotationX", q, 2.0 * b))
    lam = psi * cut
    cost = float((lam.real * psi.real + lam.imag * psi.imag).sum())
    dg, db = np.zeros(case["p"]), np.zeros(case["p"])
    for k in reversed(range(case["p"])):
        for q in range(n):
            l, x = _pairs(lam, q), _pairs(psi, q)
            db[k] += 2.0 * (_im(l[0], x[1]) + _im(l[1], x[0]))
            _apply(psi, ("ApplyRotationX", q, -2.0 * betas[k]))
            _apply(lam, ("ApplyRotationX", q, -2.0 * betas[k]))
        dg[k] = 2.0 * _im(lam, psi * cut)
        phase = torch.polar(torch.ones_like(cut), gammas[k] * cut)
        psi.mul_(phase)
        lam.mul_(phase)
    return dict(cost=np.array([cost]), gammas=dg, betas=db)


def _exact_hea(case, seed):
    costs, grads, at = [], [], 0
    angles = _hea_angles(case, seed)
    for n, d in zip(*_hea_sizes(case)):
        a = angles[at:at + 2 * n * d].reshape(d, n, 2)
        at += 2 * n * d
        sign = torch.ones(1 << n, dtype=torch.float64, device="cuda")
        for q in range(n - 1):
            _quads(sign, q + 1, q)[1][1].neg_()
        z = torch.zeros(1 << n, dtype=torch.float64, device="cuda")
        for q in range(n):
            _pairs(z, q)[0].add_(1.0)
            _pairs(z, q)[1].sub_(1.0)

        def turn(v, layer, back):
            """The diagonal of the layer's RZ rotations (and its inverse)."""
            ph = torch.zeros(1 << n, dtype=torch.float64, device="cuda")
            for q in range(n):
                lo, hi = _pairs(ph, q)
                lo.sub_(0.5 * a[layer, q, 1])
                hi.add_(0.5 * a[layer, q, 1])
            return v.mul_(torch.polar(torch.ones_like(ph), -ph if back else ph))

        def rotate(v, q, angle):
            x, y = _pairs(v, q)
            c, s = math.cos(angle / 2), math.sin(angle / 2)
            t = x * c - y * s
            y.mul_(c).add_(x, alpha=s)
            x.copy_(t)

        psi = torch.zeros(1 << n, dtype=torch.complex128, device="cuda")
        psi[0] = 1.0
        for k in range(d):
            for q in range(n):
                rotate(psi, q, a[k, q, 0])
            turn(psi, k, False).mul_(sign)
        lam = psi * z
        costs.append(float((lam.real * psi.real + lam.imag * psi.imag).sum()))
        g = torch.zeros(d, n, 2, dtype=torch.float64, device="cuda")
        for k in reversed(range(d)):
            psi.mul_(sign)
            lam.mul_(sign)
            w = lam.real * psi.imag - lam.imag * psi.real
            for q in range(n):
                lo, hi = _pairs(w, q)
                g[k, q, 1] = lo.sum() - hi.sum()
            turn(psi, k, True)
            turn(lam, k, True)
            for q in range(n):
                l, x = _pairs(lam, q), _pairs(psi, q)
                # <lam| Y |psi> = -i conj(l0) x1 + i conj(l1) x0
                g[k, q, 0] = ((l[1].real * x[0].real + l[1].imag * x[0].imag).sum() -
                              (l[0].real * x[1].real + l[0].imag * x[1].imag).sum())
                rotate(psi, q, -a[k, q, 0])
                rotate(lam, q, -a[k, q, 0])
        grads.append(g.cpu().numpy().reshape(-1))
    return dict(cost=np.array(costs), grad=np.concatenate(grads))


def _exact_readout(case, seed):
    n = case["n"]
    psi = _amplitudes(case, seed).to(torch.complex128)
    other = _amplitudes(case, seed + 1000003).to(torch.complex128)
    order = _order(n, seed)  # qubit q moves to position order[q]

    def value(qubits, observables):
        """<P> for a Pauli string: flips of the X and Y qubits, signs of the Y and Z ones."""
        t = psi
        for q, o in zip(qubits, observables):
            v = t.view(-1, 2, 1 << q)
            if o == 1:
                v = v.flip(1)
            elif o == 2:
                v = torch.stack((-1j * v[:, 1], 1j * v[:, 0]), 1)
            else:
                v = torch.stack((v[:, 0], -v[:, 1]), 1)
            t = v.reshape(-1)
        return float((psi.real * t.real + psi.imag * t.imag).sum())

    p = psi.real.square() + psi.imag.square()
    norm = float(p.sum())
    # Single-qubit values are 1 - 2 P(1) in the observable's basis; P(1) = (norm - <X>) / 2.
    x = [1.0 - (norm - value([q], [1])) for q in range(n)]
    z = [float(_pairs(p, q)[1].sum()) for q in range(n)]
    zz = []
    for a, b in _bonds(case):
        k = _quads(p, a, b)
        zz.append(float(k[0][0].sum() + k[1][1].sum() - k[0][1].sum() - k[1][0].sum()))
    strings = [value(q, o) for q, o in _correlators(n)]
    overlap = [float((other.real * psi.real + other.imag * psi.imag).sum()),
               float((other.real * psi.imag - other.imag * psi.real).sum())]
    at = list(range(n))  # the qubit at each position
    for q, position in sorted(enumerate(order), key=lambda e: e[1]):
        if at[position] != q:
            source = at.index(q)
            _apply(psi, ("ApplySwap", position, source))
            at[position], at[source] = at[source], at[position]
    return dict(x=np.array(x), z=np.array(z), zz=np.array(zz), strings=np.array(strings),
                norm=np.array([math.sqrt(norm)]), overlap=np.array(overlap), state=psi)


def exact(case, seed):
    kind = case["kind"]
    if kind == "pool":
        return None  # the noise gates' angles come from the pool's own random streams
    if kind == "qaoa":
        return _exact_qaoa(case, seed)
    if kind == "hea":
        return _exact_hea(case, seed)
    if kind == "readout":
        return _exact_readout(case, seed)
    psi = _amplitudes(case, seed).to(torch.complex128)
    for op in _ops(case, seed):
        _apply(psi, op)
    return psi
