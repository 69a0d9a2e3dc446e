"""Pool of states (intelqs_py.StatePool over iqsh_pool_*): the single-GPU form of the
reference's pool, one state per MPI rank group (src/mpi_env.cpp:239-404).

  * Trajectories: the noisy-pool tutorial's program (tutorials/get_started_with_noisy_IQS
    .cpp) on 5 states; state s must equal the compiled reference run with seed + s
    (tests/golden/pool_dp_*: same state stream as the reference's pool state s) to 1e-12,
    read-outs per state to 1e-12, the incoherent sum to their sum.
  * Common gates on Register() act on every state as on a lone register (the oracle runs
    the same gate list), padding states stay zero.
  * Per-state reductions equal numpy on the downloaded states; per-state 1- and 2-qubit
    channel branches equal ApplyChannel on a lone register seeded as that pool state."""
import os

import numpy as np
import pytest

import oracle
from iqs_amd.circuits import Circuit

pytestmark = pytest.mark.gpu
GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


def _m():
    import intelqs_py
    return intelqs_py


def _run_pool_program(pool, c):
    reg = pool.Register()
    out = []
    for op in c.ops:
        name, args = op[0], op[1:]
        if name == "SetRngSeed":
            continue  # the pool seeds every state at once
        if name in ("SetNoiseTimescales", "ApplyNoiseGate"):
            getattr(pool, name)(*args)
        elif name == "GetProbability":
            out.append((args[0], pool.GetProbability(args[0])))
        else:
            getattr(reg, name)(*args)
    return out


def test_pool_trajectories_match_reference():
    c = Circuit.parse(open(os.path.join(GOLDEN, "pool_dp.poolcirc")).read())
    ref = np.load(os.path.join(GOLDEN, "pool_dp_states.npz"))
    states, seed = ref["states"], int(ref["seed"])
    m = _m()
    pool = m.StatePool(c.num_qubits, len(states))
    pool.SetSeedStreamPtrs(seed)
    out = _run_pool_program(pool, c)
    for s in range(len(states)):
        assert np.max(np.abs(pool.GetState(s) - states[s])) < 1e-12, s
    want = {}
    for block in open(os.path.join(GOLDEN, "pool_dp.poolres")).read().split("# state ")[1:]:
        lines = block.splitlines()
        s = int(lines[0])
        for l in lines[1:]:
            t = l.split()
            want.setdefault(int(t[2]), [None] * len(states))[s] = float(t[3])
    for q, probs in out:
        assert np.max(np.abs(np.array(probs) - np.array(want[q]))) < 1e-12
        assert abs(m.StatePool.IncoherentSumOverAllStatesOfPool(probs) - sum(want[q])) < 1e-12
    # Padding states (5 of 8 slots used) are untouched.
    full = np.array(pool.Register(), copy=True)
    assert np.all(full[len(states) << c.num_qubits:] == 0)


def test_common_gates_act_on_every_state():
    m = _m()
    n, k = 7, 3
    pool = m.StatePool(n, k, "++++", 0)
    c = Circuit(n, precision="dp", init="plus")
    rs = np.random.default_rng(17)
    for _ in range(30):
        q = int(rs.integers(n))
        kind = int(rs.integers(4))
        if kind == 0:
            c.add("ApplyRotationX", q, float(rs.uniform(0, 6)))
        elif kind == 1:
            c.add("ApplyHadamard", q)
        elif kind == 2:
            c.add("ApplyCPauliX", q, (q + 1 + int(rs.integers(n - 1))) % n)
        else:
            c.add("ApplySwap", q, (q + 2) % n)
    reg = pool.Register()
    for op in c.ops:
        getattr(reg, op[0])(*op[1:])
    want, _ = oracle.run(c.to_text())
    for s in range(k):
        assert np.max(np.abs(pool.GetState(s) - want)) < 1e-12, s
    assert np.allclose(pool.ComputeNorm(), 1.0, atol=1e-12)


def test_per_state_reductions_and_overlap():
    c = Circuit.parse(open(os.path.join(GOLDEN, "pool_dp.poolcirc")).read())
    m = _m()
    ns = 6
    pool = m.StatePool(c.num_qubits, ns)
    pool.SetSeedStreamPtrs(99)
    _run_pool_program(pool, c)
    pool.Register().ApplyHadamard(2)
    st = [pool.GetState(s) for s in range(ns)]
    idx = np.arange(st[0].size)
    for q in (0, 4):
        want = [np.sum(np.abs(v[(idx >> q) & 1 == 1]) ** 2) for v in st]
        assert np.max(np.abs(np.array(pool.GetProbability(q)) - want)) < 1e-13
    mask = (1 << 1) | (1 << 5)
    sign = np.where(np.array([bin(i & mask).count("1") & 1 for i in idx]) == 1, -1.0, 1.0)
    want = [np.sum(sign * np.abs(v) ** 2) for v in st]
    assert np.max(np.abs(np.array(pool.ExpectationValueZString([1, 5])) - want)) < 1e-13
    assert np.max(np.abs(np.array(pool.ComputeNorm()) - [np.linalg.norm(v) for v in st])) < 1e-13
    ideal = m.QubitRegister(c.num_qubits, "base", 0, 0)
    ideal.ApplyHadamard(0)
    ideal.ApplyRotationY(3, 0.7)
    iv = np.array(ideal, copy=True)
    got = pool.ComputeOverlap(ideal)
    want = [np.vdot(iv, v) for v in st]
    assert np.max(np.abs(np.array(got) - want)) < 1e-13


def test_per_state_channel_matches_lone_registers():
    m = _m()
    n, ns, seed = 5, 4, 31
    chi = np.diag([0.6, 0.25, 0.1, 0.05]).astype(complex)
    cm = m.CM4x4(chi)
    cm.SolveEigenSystem()
    pool = m.StatePool(n, ns, "++++", 0)
    pool.SetSeedStreamPtrs(seed)
    for step in range(6):
        pool.ApplyChannel(step % n, cm)
        pool.Register().ApplyCPauliX(step % n, (step + 2) % n)
    for s in range(ns):
        reg = m.QubitRegister(n, "++++", 0, 0)
        rng = m.RandomNumberGenerator()
        rng.SetSeedStreamPtrs(seed + s)  # its state stream is pool state s's
        reg.SetRngPtr(rng)
        for step in range(6):
            reg.ApplyChannel(step % n, cm)
            reg.ApplyCPauliX(step % n, (step + 2) % n)
        reg.ResetRngPtr()
        assert np.max(np.abs(pool.GetState(s) - np.array(reg, copy=True))) < 1e-12, s


@pytest.mark.parametrize("order", ["high_first", "low_first"])
def test_per_state_2q_channel_matches_lone_registers(order):
    """2-qubit channel branches (a dense complex chi, so every Pauli pair term is present)
    drawn per state; both qubit orders pin the 2 b(qubit1) + b(qubit2) row convention of
    the per-state kernel against Apply2QubitGate.  Three states: the padding state stays 0."""
    m = _m()
    n, ns, seed = 6, 3, 57
    r = np.random.default_rng(12)
    a = r.normal(size=(16, 16)) + 1j * r.normal(size=(16, 16))
    chi = a @ a.conj().T
    chi /= np.trace(chi).real
    cm = m.CM16x16(chi)
    cm.SolveEigenSystem()
    pairs = [(4, 1), (0, 5), (3, 2)] if order == "high_first" else [(1, 4), (5, 0), (2, 3)]
    pool = m.StatePool(n, ns, "++++", 0)
    pool.SetSeedStreamPtrs(seed)
    for step in range(5):
        q1, q2 = pairs[step % 3]
        pool.ApplyChannel(q1, q2, cm)
        pool.Register().ApplyRotationY(step % n, 0.3 + step)
    signs = pool.GetOverallSignOfChannels()
    for s in range(ns):
        reg = m.QubitRegister(n, "++++", 0, 0)
        rng = m.RandomNumberGenerator()
        rng.SetSeedStreamPtrs(seed + s)
        reg.SetRngPtr(rng)
        for step in range(5):
            q1, q2 = pairs[step % 3]
            reg.ApplyChannel(q1, q2, cm)
            reg.ApplyRotationY(step % n, 0.3 + step)
        reg.ResetRngPtr()
        want = np.array(reg, copy=True)
        assert np.max(np.abs(want)) > 1e-3
        assert np.max(np.abs(pool.GetState(s) - want)) < 1e-12, s
        assert signs[s] == reg.GetOverallSignOfChannels()
    full = np.array(pool.Register(), copy=True)
    assert np.all(full[ns << n:] == 0)
    with pytest.raises(ValueError):
        pool.ApplyChannel(2, 2, cm)


def test_pool_errors():
    m = _m()
    pool = m.StatePool(4, 3)
    with pytest.raises(IndexError):
        pool.GetProbability(4)
    with pytest.raises(IndexError):
        pool.GetState(3)
    with pytest.raises(ValueError):
        m.StatePool(4, 0)
    with pytest.raises(ValueError):
        pool.Initialize("rand", 0)
    with pytest.raises(ValueError):
        m.MPIEnvironment.UpdateStateComm(4)


@pytest.mark.parametrize("dt", ["c128", "c64"])
def test_per_state_kernels_every_form(dt):
    """iqsh_pool_* on 9-qubit states (3 states in 4 slots, the fourth left as uploaded):
    per-state 1q at positions below 6 (lane-shuffle form) and from 6 up (pair tiles), per-state
    2q with both positions inside a 128-byte line and outside it, then every per-state
    reduction, each against numpy on the same states."""
    import ctypes as C

    from iqs_amd._lib import call
    from iqs_amd.circuits import SplitMix64, haar_unitary
    from iqs_amd.engine import StateVector

    sq, ns, n = 9, 3, 11
    npdt = np.complex128 if dt == "c128" else np.complex64
    tol = 1e-12 if dt == "c128" else 2e-5
    r = np.random.default_rng(61)
    host = (r.normal(size=1 << n) + 1j * r.normal(size=1 << n)).astype(npdt)
    sv = StateVector(n, dt)
    sv.upload(host)
    want = host.astype(np.complex128).reshape(1 << (n - sq), 1 << sq)
    rng = SplitMix64(62)

    def mats(k):
        us = [haar_unitary(1 << k, rng) for _ in range(ns)]
        flat = np.concatenate([np.stack([u.real, u.imag], -1).reshape(-1) for u in us]).astype(np.float64)
        return us, flat

    for pos in (0, 3, 5, 6, 8):
        us, flat = mats(1)
        call("iqsh_pool_apply_1q_each", sv.handle, sq, pos, flat.ctypes.data_as(C.POINTER(C.c_double)), ns)
        for s in range(ns):
            v = want[s].reshape(1 << (sq - 1 - pos), 2, 1 << pos)
            want[s] = np.einsum("ij,ajb->aib", us[s].astype(npdt).astype(np.complex128), v).reshape(-1)
    idx = np.arange(1 << sq)
    for ph, pl in ((1, 0), (2, 7), (8, 6)):
        us, flat = mats(2)
        call("iqsh_pool_apply_2q_each", sv.handle, sq, ph, pl, flat.ctypes.data_as(C.POINTER(C.c_double)), ns)
        base = idx[((idx >> ph) & 1) == 0]
        base = base[((base >> pl) & 1) == 0]
        rows = [base, base | (1 << pl), base | (1 << ph), base | (1 << ph) | (1 << pl)]
        for s in range(ns):
            x = np.stack([want[s][rw] for rw in rows])
            y = us[s].astype(npdt).astype(np.complex128) @ x
            for t, rw in enumerate(rows):
                want[s][rw] = y[t]
    got = sv.download().astype(np.complex128).reshape(1 << (n - sq), 1 << sq)
    assert np.abs(got[:ns] - want[:ns]).max() < tol
    assert np.array_equal(got[ns:], host.astype(np.complex128).reshape(1 << (n - sq), 1 << sq)[ns:])
    out = (C.c_double * (2 * ns))()
    for kind, arg, f in ((0, 0, lambda v: np.sum(np.abs(v) ** 2)),
                         (1, 4, lambda v: np.sum(np.abs(v[(idx >> 4) & 1 == 1]) ** 2)),
                         (2, 0b100010001, lambda v: np.sum(np.where(
                             np.array([bin(i & 0b100010001).count("1") & 1 for i in idx]) == 1, -1.0, 1.0)
                             * np.abs(v) ** 2))):
        call("iqsh_pool_reduce", sv.handle, sq, kind, arg, out, ns)
        assert np.max(np.abs(np.array(out[:ns]) - [f(got[s]) for s in range(ns)])) < 1e-11
    ref_h = (r.normal(size=1 << sq) + 1j * r.normal(size=1 << sq)).astype(npdt)
    ref = StateVector(sq, dt)
    ref.upload(ref_h)
    call("iqsh_pool_overlap", sv.handle, sq, ref.handle, out, ns)
    wov = [np.vdot(ref_h.astype(np.complex128), got[s]) for s in range(ns)]
    assert np.max(np.abs(np.array(out[0::2]) + 1j * np.array(out[1::2]) - wov)) < 1e-11


@pytest.mark.parametrize("dt", ["c128", "c64"])
@pytest.mark.parametrize("sbits,nstates", [(3, 5), (9, 3), (11, 2), (12, 7), (14, 33), (15, 3), (16, 40)])
def test_per_state_matrices_and_probabilities_over_sizes(dt, sbits, nstates):
    """Matrices in the kernel's arguments and in the slot ring (more of them than 2048 bytes
    hold, several calls in a row), chunks of every size, and P(qubit) on every position, against
    numpy on the host.  Tolerances: one 2x2 product per call (4 roundings), sums of at most 2^16
    terms in FP64."""
    import ctypes as C

    from iqs_amd._lib import call
    from iqs_amd.engine import StateVector
    n = sbits + max(1, (nstates - 1).bit_length())
    r = np.random.default_rng(sbits)
    v = r.normal(size=1 << n) + 1j * r.normal(size=1 << n)
    v = (v / np.linalg.norm(v)).astype(np.complex128 if dt == "c128" else np.complex64)
    sv = StateVector(n, dt)
    sv.upload(v)
    want = v.astype(np.complex128).reshape(-1, 1 << sbits)
    for call_no in range(6):
        pos = (call_no * 5) % sbits
        th = r.uniform(0, 6, nstates)
        m = np.zeros((nstates, 2, 2), dtype=np.complex128)
        m[:, 0, 0] = m[:, 1, 1] = np.cos(th)
        m[:, 0, 1], m[:, 1, 0] = -np.sin(th), np.sin(th)
        call("iqsh_pool_apply_1q_each", sv.handle, C.c_uint(sbits), C.c_uint(pos), C.c_void_p(m.ctypes.data), C.c_uint64(nstates))
        w = want[:nstates].reshape(nstates, -1, 2, 1 << pos)
        a, b = w[:, :, 0].copy(), w[:, :, 1].copy()
        w[:, :, 0] = m[:, 0, 0, None, None] * a + m[:, 0, 1, None, None] * b
        w[:, :, 1] = m[:, 1, 0, None, None] * a + m[:, 1, 1, None, None] * b
    got = sv.download().reshape(-1, 1 << sbits)
    eps = 2.0 ** -52 if dt == "c128" else 2.0 ** -23
    assert np.abs(got - want).max() < 6 * 4 * eps * np.abs(v).max() * 2
    assert np.array_equal(got[nstates:], v.reshape(-1, 1 << sbits)[nstates:])
    p = np.abs(got.astype(np.complex128)) ** 2
    out = np.zeros(nstates)
    for pos in range(sbits):
        call("iqsh_pool_reduce", sv.handle, C.c_uint(sbits), C.c_int(1), C.c_uint64(pos), C.c_void_p(out.ctypes.data),
             C.c_uint64(nstates))
        assert np.abs(out - p[:nstates].reshape(nstates, -1, 2, 1 << pos)[:, :, 1].sum(axis=(1, 2))).max() < 1e-13
    call("iqsh_pool_reduce", sv.handle, C.c_uint(sbits), C.c_int(0), C.c_uint64(0), C.c_void_p(out.ctypes.data),
         C.c_uint64(nstates))
    assert np.abs(out - p[:nstates].sum(axis=1)).max() < 1e-13


@pytest.mark.parametrize("dt", ["c128", "c64"])
@pytest.mark.parametrize("sbits,nstates", [(3, 8192), (3, 8193), (3, 70000), (12, 4097), (9, 9000)])
def test_reductions_over_many_states(dt, sbits, nstates):
    """Sums written to the host by the kernels (up to 8192 workgroups) and copied from the device
    (more), around the limit and far beyond it, one and two values per workgroup, against numpy.
    Tolerance: sums of at most 2^12 products in FP64, of states of norm 1."""
    import ctypes as C

    from iqs_amd._lib import call
    from iqs_amd.engine import StateVector
    n = sbits + (nstates - 1).bit_length()
    r = np.random.default_rng(nstates)
    v = r.standard_normal((1 << (n - sbits), 1 << sbits)) + 1j * r.standard_normal((1 << (n - sbits), 1 << sbits))
    v = (v / np.linalg.norm(v, axis=1, keepdims=True)).astype(np.complex128 if dt == "c128" else np.complex64)
    sv, ref = StateVector(n, dt), StateVector(sbits, dt)
    sv.upload(v.reshape(-1))
    ref.upload(v[1])
    w = v.astype(np.complex128)[:nstates]
    p = np.abs(w) ** 2
    sign = np.array([1 - 2 * (bin(i & 5).count("1") & 1) for i in range(1 << sbits)])
    top = sbits - 1
    out = np.zeros(2 * nstates)
    for kind, arg, want in ((0, 0, p.sum(1)), (1, 0, p.reshape(nstates, -1, 2)[:, :, 1].sum(1)),
                            (1, top, p[:, 1 << top:].sum(1)), (2, 5, (p * sign).sum(1))):
        call("iqsh_pool_reduce", sv.handle, C.c_uint(sbits), C.c_int(kind), C.c_uint64(arg), C.c_void_p(out.ctypes.data),
             C.c_uint64(nstates))
        assert np.abs(out[:nstates] - want).max() < 1e-13
    call("iqsh_pool_overlap", sv.handle, C.c_uint(sbits), ref.handle, C.c_void_p(out.ctypes.data), C.c_uint64(nstates))
    assert np.abs(out.view(np.complex128) - w @ w[1].conj()).max() < 1e-13


def test_per_state_matrices_in_a_capture():
    """Matrices that fit a kernel's arguments can be captured into a graph and are replayed as they
    were; more of them (a slot that later calls refill) are refused, and the capture goes on."""
    import ctypes as C

    torch = pytest.importorskip("torch")
    from iqs_amd._lib import IqsError, call
    from iqs_amd.engine import StateVector
    sbits, n = 5, 12
    sv, want = StateVector(n, "c128"), StateVector(n, "c128")

    def rotations(ns, seed):
        th = np.random.default_rng(seed).uniform(0, 6, ns)
        m = np.zeros((ns, 2, 2), dtype=np.complex128)
        m[:, 0, 0] = m[:, 1, 1] = np.cos(th)
        m[:, 0, 1], m[:, 1, 0] = -np.sin(th), np.sin(th)
        return m

    def each(target, m):
        call("iqsh_pool_apply_1q_each", target.handle, C.c_uint(sbits), C.c_uint(3), C.c_void_p(m.ctypes.data), C.c_uint64(len(m)))

    few, many = rotations(30, 1), rotations(100, 2)
    for v in (sv, want):
        v.init_uniform(2.0 ** (-n / 2))
        each(v, many)
    call("iqsh_sync")
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    try:
        call("iqsh_set_stream", C.c_void_p(stream.cuda_stream))
        with torch.cuda.graph(graph, stream=stream):
            with pytest.raises(IqsError):
                each(sv, many)
            each(sv, few)
        for k in range(3):
            with torch.cuda.stream(stream):
                graph.replay()
            each(want, few)
            assert sv.maxabsdiff(want) < 1e-14
            each(sv, many)
            each(want, many)
            assert sv.maxabsdiff(want) < 1e-14
    finally:
        call("iqsh_sync")
        call("iqsh_set_stream", None)


@pytest.mark.parametrize("dt", ["c128", "c64"])
def test_matrix_slots_grow_between_streams(dt):
    """Per-state 2x2 and 4x4 matrices of pools that take turns, each larger one growing the slots while
    the launches of the one before are still on another stream: 2x2 in arguments and slots for both
    precisions, 4x4 likewise, against numpy.  Tolerance: one product of two or four terms per call and
    amplitude (8 roundings of amplitudes below 8), three calls."""
    import ctypes as C

    torch = pytest.importorskip("torch")
    from iqs_amd._lib import call
    from iqs_amd.circuits import SplitMix64, haar_unitary
    from iqs_amd.engine import StateVector
    npdt = np.complex128 if dt == "c128" else np.complex64
    tol = 3 * 8 * 8 * (2.0 ** -53 if dt == "c128" else 2.0 ** -24)
    rng, r = SplitMix64(3), np.random.default_rng(4)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    pools = []
    try:
        for k, (sbits, ns) in enumerate([(12, 9), (6, 66), (11, 17), (5, 300), (10, 40), (4, 2000), (9, 100), (4, 9000)]):
            n = sbits + (ns - 1).bit_length()
            host = (r.uniform(-1, 1, 1 << n) + 1j * r.uniform(-1, 1, 1 << n)).astype(npdt)
            want = host.astype(np.complex128).reshape(-1, 1 << sbits)
            call("iqsh_set_stream", C.c_void_p(streams[k % 2].cuda_stream))
            sv = StateVector(n, dt)
            sv.upload(host)
            for pos in ((sbits - 1,), (2, 0), (1, sbits - 1)):
                d = 1 << len(pos)
                few = [haar_unitary(d, rng) for _ in range(min(ns, 50))]
                us = np.stack([few[s % len(few)] * np.exp(1j * s) for s in range(ns)]).astype(npdt).astype(np.complex128)
                name = "iqsh_pool_apply_1q_each" if d == 2 else "iqsh_pool_apply_2q_each"
                call(name, sv.handle, C.c_uint(sbits), *(C.c_uint(p) for p in pos), C.c_void_p(us.ctypes.data), C.c_uint64(ns))
                i = np.arange(1 << sbits)
                base = i[sum((i >> p) & 1 for p in pos) == 0]
                rows = [base + sum(((t >> (len(pos) - 1 - j)) & 1) << p for j, p in enumerate(pos)) for t in range(d)]
                x = np.stack([want[:ns][:, rw] for rw in rows], 1)
                y = us @ x
                for t, rw in enumerate(rows):
                    want[:ns, rw] = y[:, t]
            pools.append((sv, want))
    finally:
        torch.cuda.synchronize()
        call("iqsh_set_stream", None)
    for sv, want in pools:
        assert np.abs(sv.download().reshape(want.shape) - want).max() < tol
