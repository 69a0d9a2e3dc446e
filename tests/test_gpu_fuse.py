"""Gate lists applied together (iqsh_apply_gates, TurnOnFusion) against the same gates one by
one on the GPU: sizes around the tile (2^10 below 12 qubits, 2^12 from there; dense blocks below
10), every block size, lists that fill more than one slot of the descriptor ring, repeated pairs
in both orders, gates on fresh and on used qubits, and the cached accesses of a 32 MiB register.
Tolerances: those of the fused-against-unfused tests (1e-12, 2e-5 absolute)."""
import ctypes as C

import numpy as np
import pytest

from iqs_amd import runner
from iqs_amd._lib import IqsError, call
from iqs_amd.circuits import Circuit, SplitMix64, haar_unitary
from iqs_amd.engine import StateVector

pytestmark = pytest.mark.gpu
TOL = {"dp": 1e-12, "sp": 2e-5}


def _mixed(n, count, seed, precision):
    """Random one- and two-qubit gates, CNOTs, repeated pairs (both orders) and rotations."""
    r = SplitMix64(seed)
    c = Circuit(n, precision=precision, init="plus")
    pair = (0, 1)
    for i in range(count):
        k = r.randint(6)
        a = r.randint(n)
        b = (a + 1 + r.randint(n - 1)) % n
        if k == 0:
            c.add("Apply1QubitGate", a, haar_unitary(2, r))
        elif k == 1:
            c.add("Apply2QubitGate", a, b, haar_unitary(4, r))
            pair = (a, b)
        elif k == 2:
            c.add("ApplyCPauliX", a, b)
        elif k == 3:
            c.add("Apply2QubitGate", pair[1], pair[0], haar_unitary(4, r))
        elif k == 4:
            c.add("ApplyRotationZ", a, r.uniform(0.0, 6.0))
        else:
            c.add("ApplyHadamard", a)
    return c


def _compare(c, block):
    ref, _ = runner.run(c)
    reg = runner.new_register(c)
    reg.SetFusionBlockQubits(block)
    reg.TurnOnFusion()
    reg, _ = runner.run(c, reg)
    assert np.abs(runner.state_of(reg) - runner.state_of(ref)).max() < TOL[c.precision]
    return reg.FusionStats()


@pytest.mark.parametrize("precision", ["dp", "sp"])
@pytest.mark.parametrize("n", [2, 5, 9, 10, 11, 12, 13, 15, 17, 21, 22])
def test_gate_lists_match_single_gates(precision, n):
    for count, seed in ((1, 3), (7, 4), (60, 5)):
        _compare(_mixed(n, count, 100 * n + seed, precision), 5)


@pytest.mark.parametrize("block", [1, 2, 3, 4])
@pytest.mark.parametrize("n", [8, 10, 14])
def test_block_sizes(n, block):
    _compare(_mixed(n, 40, n + block, "dp"), block)


def test_long_lists_take_several_launches():
    gates, passes = _compare(_mixed(12, 900, 8, "dp"), 5)
    assert gates == 900 and passes >= 2  # one tile, more blocks than one launch holds
    _compare(_mixed(14, 900, 9, "sp"), 5)


def test_bad_gate_lists_are_refused():
    class Gate(C.Structure):
        _fields_ = [("np", C.c_uint), ("p", C.c_uint * 2), ("m", C.c_double * 32)]

    sv = StateVector(11, "c128")
    sv.init_basis(3)
    passes = C.c_uint64(7)
    call("iqsh_apply_gates", sv.handle, 0, None, 5, C.byref(passes))
    assert passes.value == 0
    for np_, p, block in ((0, (0, 1), 5), (3, (0, 1), 5), (1, (11, 0), 5), (2, (4, 4), 5), (2, (0, 1), 0), (2, (0, 1), 6)):
        g = Gate(np_, (C.c_uint * 2)(*p))
        with pytest.raises(IqsError):
            call("iqsh_apply_gates", sv.handle, 1, C.byref(g), block, None)
    assert sv.prob1(0) == 1.0 and sv.norm2() == 1.0


@pytest.mark.parametrize("seed", [1, 2])
def test_double_precision_error_of_merged_gates(seed):
    """Forty brick layers of 14 qubits (H, rotation, CNOT ladder; 74 blocks of 4 positions,
    96 allowed for) against the same gates in 80-bit arithmetic.  Tolerance (2-norm of a state of norm 1): a block
    rounds its matrix and, per amplitude, sums of 16 terms in three real products, 6 units of 2^-53 at
    most, independent from block to block: sqrt(96) * 6 * 2^-53.  (Roundings that all amplitudes
    share add up with the number of gates instead.)"""
    from iqs_amd import gates as G
    n, r = 14, SplitMix64(seed)
    c = Circuit(n, precision="dp", init="plus")
    want = np.full(1 << n, 2.0 ** (-n / 2), dtype=np.clongdouble)
    for layer in range(40):
        mats = [(q, m) for rnd in (lambda: G.H, lambda: (G.rx, G.ry, G.rz)[r.randint(3)](r.uniform(0.0, 6.28)))
                for q in range(n) for m in (rnd(),)]
        for q, m in mats:
            c.add("Apply1QubitGate", q, m)
            v = want.reshape(-1, 2, 1 << q)
            m = m.astype(np.clongdouble)
            v[:, 0], v[:, 1] = m[0, 0] * v[:, 0] + m[0, 1] * v[:, 1], m[1, 0] * v[:, 0] + m[1, 1] * v[:, 1]
        for q in range(layer % 2, n - 1, 2):
            c.add("ApplyCPauliX", q, q + 1)
            v = want.reshape(-1, 2, 2, 1 << q)
            v[:, :, 1] = v[:, ::-1, 1].copy()
    reg = runner.new_register(c)
    reg.TurnOnFusion()
    reg, _ = runner.run(c, reg)
    err = float(np.sqrt(np.sum(np.abs(runner.state_of(reg) - want) ** 2)))
    print(f"brick 14 x 40, seed {seed}: error {err:.2e}", flush=True)
    assert err < 96 ** 0.5 * 6 * 2.0 ** -53


@pytest.mark.parametrize("dt", ["c128", "c64"])
@pytest.mark.parametrize("mode", [0, 2])
def test_chosen_block_kernel_applies_gate_lists(dt, mode):
    """With a block kernel chosen (iqsh_set_block_mfma), a list on five positions is one pass of that
    kernel: the same bits as iqsh_apply_kq with the product, which is exact for these entries."""
    class Gate(C.Structure):
        _fields_ = [("np", C.c_uint), ("p", C.c_uint * 2), ("m", C.c_double * 32)]

    n, pos = 13, [1, 4, 6, 9, 12]
    r = np.random.default_rng(mode)
    v = r.normal(size=1 << n) + 1j * r.normal(size=1 << n)
    v = (v / np.linalg.norm(v)).astype(np.complex128 if dt == "c128" else np.complex64)
    ms = [r.choice([0.5, -0.5, 0.5j, -0.25j, 0.75], (2, 2)) for _ in pos]
    u = np.ones((1, 1), dtype=np.complex128)
    gates = (Gate * 5)()
    for i, (p, m) in enumerate(zip(pos, ms)):
        u = np.kron(m, u)  # index bit i <-> pos[i]
        gates[i].np, gates[i].p[0] = 1, p
        gates[i].m[:8] = np.ascontiguousarray(m).view(np.float64).reshape(-1).tolist()
    a, b, passes = StateVector(n, dt), StateVector(n, dt), C.c_uint64()
    a.upload(v)
    b.upload(v)
    u = np.ascontiguousarray(u)
    call("iqsh_set_block_mfma", mode)
    try:
        call("iqsh_apply_gates", a.handle, 5, gates, 5, C.byref(passes))
        call("iqsh_apply_kq", b.handle, 5, (C.c_uint * 5)(*pos), C.c_void_p(u.ctypes.data))
    finally:
        call("iqsh_set_block_mfma", 1)
    assert passes.value == 1
    assert np.array_equal(a.download(), b.download())


@pytest.mark.parametrize("block", [2, 5])
@pytest.mark.parametrize("dt", ["c128", "c64"])
def test_captured_gate_lists_replay_their_own_gates(dt, block):
    """A list captured into a graph, replayed between and after other lists (which use every slot of
    the ring again), against the same list applied without a graph: three times the roundings of
    the fused-against-unfused tests."""
    torch = pytest.importorskip("torch")

    class Gate(C.Structure):
        _fields_ = [("np", C.c_uint), ("p", C.c_uint * 2), ("m", C.c_double * 32)]

    def gates(seed, count):
        r = SplitMix64(seed)
        out = (Gate * count)()
        for g in out:
            a = r.randint(n)
            g.np, g.p[0], g.p[1] = 2, a, (a + 1 + r.randint(n - 1)) % n
            g.m[:] = haar_unitary(4, r).astype(np.complex128).view(np.float64).reshape(-1).tolist()
        return out

    n, count = 13, 12
    one = gates(1, count)
    a, b, other = (StateVector(n, dt) for _ in range(3))
    for sv in (a, b, other):
        sv.init_uniform(2.0 ** (-n / 2))
    call("iqsh_apply_gates", other.handle, count, one, block, None)  # buffers exist
    call("iqsh_sync")
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    stream.wait_stream(torch.cuda.current_stream())
    try:
        call("iqsh_set_stream", C.c_void_p(stream.cuda_stream))
        with torch.cuda.graph(graph, stream=stream):
            call("iqsh_apply_gates", a.handle, count, one, block, None)
        for k in range(3):
            for i in range(5):
                call("iqsh_apply_gates", other.handle, count, gates(10 * k + i + 2, count), block, None)
            call("iqsh_sync")
            with torch.cuda.stream(stream):
                graph.replay()
            call("iqsh_apply_gates", b.handle, count, one, block, None)
            call("iqsh_sync")
            assert np.abs(a.download() - b.download()).max() < 3 * TOL["dp" if dt == "c128" else "sp"]
    finally:
        call("iqsh_sync")
        call("iqsh_set_stream", None)


@pytest.mark.parametrize("dt,n", [("c128", 22), ("c64", 23)])
def test_many_gates_on_five_qubits_are_one_block(dt, n):
    """Many gates on five positions of a large register are one dense block (not a pass of many
    smaller ones): the same bits as iqsh_apply_kq with the product, which is exact for these
    gates (permutations with phases of +-1 and +-i, one term per row and so the same sums in any
    order).  A block of four positions at most rounds again in between."""
    class Gate(C.Structure):
        _fields_ = [("np", C.c_uint), ("p", C.c_uint * 2), ("m", C.c_double * 32)]

    count, pos = 60, [2, 7, 11, 16, n - 1]
    r = np.random.default_rng(n)
    u = np.eye(32, dtype=np.complex128)
    gates = (Gate * count)()
    for g in gates:
        a, b = (int(x) for x in r.choice(5, 2, replace=False))
        m = np.eye(4)[r.permutation(4)] * r.choice([1, -1, 1j, -1j], 4)[:, None]
        g.np, g.p[0], g.p[1] = 2, pos[a], pos[b]
        g.m[:] = m.astype(np.complex128).view(np.float64).reshape(-1).tolist()
        i = np.arange(32)
        sub = 2 * ((i >> a) & 1) + ((i >> b) & 1)
        rest = i & ~((1 << a) | (1 << b))
        u = (m[np.ix_(sub, sub)] * (rest[:, None] == rest[None, :])) @ u
    v = (r.standard_normal(1 << n) + 1j * r.standard_normal(1 << n)) * 2.0 ** (-n / 2)
    a, b, passes = StateVector(n, dt), StateVector(n, dt), C.c_uint64()
    a.upload(v.astype(np.complex128 if dt == "c128" else np.complex64))
    b.copy_from(a)
    u = np.ascontiguousarray(u)
    call("iqsh_apply_kq", b.handle, 5, (C.c_uint * 5)(*pos), C.c_void_p(u.ctypes.data))
    call("iqsh_apply_gates", a.handle, count, gates, 5, C.byref(passes))
    assert passes.value == 1 and a.maxabsdiff(b) == 0.0
