"""Layers of one gate on every qubit (iqsh_apply_1q_all / iqsh_adjoint_1q_all): the forward
layer against the oracle applying the gate qubit by qubit (tiles of 2^10 to 2^13 amplitudes, by
size and precision; one to three passes); the adjoint layer against the
per-qubit adjoint step on the GPU and against sum_q 2 Im <lam| G_q |psi> computed with the
oracle's 1q kernel on the host (G_q psi for each q), then the oracle's per-qubit undo."""
import numpy as np
import pytest

import oracle
from iqs_amd.circuits import SplitMix64
from iqs_amd._lib import IqsError
from iqs_amd.engine import StateVector

pytestmark = pytest.mark.gpu
TOL = {"c128": 1e-12, "c64": 1e-5}
DT = {"c128": np.complex128, "c64": np.complex64}


def _state(n, dt, seed):
    r = np.random.default_rng(seed)
    v = r.normal(size=1 << n) + 1j * r.normal(size=1 << n)
    return (v / np.linalg.norm(v)).astype(DT[dt])


def _unitary(seed):
    r = SplitMix64(seed)
    a, b, c = (r.uniform(0, 6.28) for _ in range(3))
    return np.array([[np.exp(1j * a) * np.cos(b), -np.exp(1j * c) * np.sin(b)],
                     [np.exp(-1j * c) * np.sin(b), np.exp(-1j * a) * np.cos(b)]])


def _gpu(h, dt):
    sv = StateVector(int(h.size).bit_length() - 1, dt)
    sv.upload(h)
    return sv


@pytest.mark.parametrize("dt", ["c128", "c64"])
@pytest.mark.parametrize("n", [10, 11, 13, 17, 20])
def test_layer_forward(dt, n):
    h = _state(n, dt, n)
    u = _unitary(100 + n)
    sv = _gpu(h, dt)
    sv.apply_1q_all(u)
    for q in range(n):
        oracle.apply_1q(h, q, u)
    assert np.abs(sv.download() - h).max() < TOL[dt]


@pytest.mark.parametrize("gen", ["general", "X"])
@pytest.mark.parametrize("dt", ["c128", "c64"])
@pytest.mark.parametrize("n", [10, 12, 15, 20])
def test_layer_adjoint(dt, n, gen):
    """Any generator, and G = X exactly (the kernels' two-product form of the term)."""
    psi = _state(n, dt, 2 * n)
    lam = _state(n, dt, 2 * n + 1)
    u = _unitary(7 * n)
    uinv = u.conj().T
    if gen == "X":
        G = np.array([[0, 1], [1, 0]], dtype=complex)
    else:
        G = np.array([[0.3, 1.2 - 0.4j], [1.2 + 0.4j, -0.7]])  # any 2x2, Hermitian here
    # reference value: sum_q 2 Im <lam| G_q |psi> on the host (FP64)
    want = 0.0
    for q in range(n):
        gp = psi.astype(np.complex128).copy()
        oracle.apply_1q(gp, q, G)
        want += 2 * np.imag(np.vdot(lam.astype(np.complex128), gp))
    a, b = _gpu(psi, dt), _gpu(lam, dt)
    got = a.adjoint_1q_all(b, uinv, G)
    # per-qubit adjoint steps on the GPU
    c, d = _gpu(psi, dt), _gpu(lam, dt)
    seq = sum(c.adjoint_1q(d, q, uinv, G) for q in reversed(range(n)))
    scale = max(1.0, abs(want))
    assert abs(got - want) < (1e-11 if dt == "c128" else 2e-5) * scale
    assert abs(got - seq) < (1e-11 if dt == "c128" else 2e-5) * scale
    hp, hl = psi.copy(), lam.copy()
    for q in range(n):
        oracle.apply_1q(hp, q, uinv)
        oracle.apply_1q(hl, q, uinv)
    assert np.abs(a.download() - hp).max() < TOL[dt]
    assert np.abs(b.download() - hl).max() < TOL[dt]
    assert np.abs(a.download() - c.download()).max() < TOL[dt]


def test_layer_needs_ten_qubits():
    sv = StateVector(9, "c128")
    with pytest.raises(IqsError):
        sv.apply_1q_all(np.eye(2))


def _graph(n, seed, weighted):
    r = np.random.default_rng(seed)
    edges = [(i, (i + 1) % n, float(r.uniform(0.3, 1.9)) if weighted else 1.0) for i in range(n)]
    edges += [(0, n // 2, 0.7 if weighted else 1.0), (1, n - 2, 1.3 if weighted else 1.0)]
    return edges


@pytest.mark.parametrize("dt", ["c128", "c64"])
@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("n", [12, 20])
def test_qaoa_layer_fused_equals_unfused(dt, weighted, n):
    """iqsh_qaoa_layer = iqsh_qaoa_phase then the mixer on every qubit; the fused adjoint =
    iqsh_adjoint_1q_all then iqsh_qaoa_phase_adjoint (gradients and states); the forward
    layer also against the oracle (cost diagonal from the edge list, 1q kernel per qubit)."""
    from iqs_amd import gates as Gt
    edges = _graph(n, 3, weighted)
    gamma, beta = 0.83, 0.41
    psi = _state(n, dt, 41)
    a, b = _gpu(psi, dt), _gpu(psi, dt)
    a.qaoa_layer(edges, gamma, Gt.rx(2 * beta))
    b.qaoa_phase(edges, gamma)
    b.apply_1q_all(Gt.rx(2 * beta))
    assert np.abs(a.download() - b.download()).max() < TOL[dt]
    h = psi.astype(np.complex128).copy()
    x = np.arange(1 << n)
    cut = sum(w * (((x >> u) ^ (x >> v)) & 1) for u, v, w in edges)
    h *= np.exp(-1j * gamma * cut)
    for q in range(n):
        oracle.apply_1q(h, q, Gt.rx(2 * beta))
    assert np.abs(a.download() - h).max() < (1e-12 if dt == "c128" else 2e-5)
    lam = _state(n, dt, 42)
    X = np.array([[0, 1], [1, 0]])
    p1, l1 = _gpu(psi, dt), _gpu(lam, dt)
    dg1, db1 = p1.qaoa_layer_adjoint(l1, edges, gamma, Gt.rx(-2 * beta), X)
    p2, l2 = _gpu(psi, dt), _gpu(lam, dt)
    db2 = p2.adjoint_1q_all(l2, Gt.rx(-2 * beta), X)
    dg2 = p2.qaoa_phase_adjoint(l2, edges, gamma)
    tol = 1e-11 if dt == "c128" else 2e-5
    assert abs(db1 - db2) < tol * max(1, abs(db2)) and abs(dg1 - dg2) < tol * max(1, abs(dg2))
    assert np.abs(p1.download() - p2.download()).max() < TOL[dt]
    assert np.abs(l1.download() - l2.download()).max() < TOL[dt]


@pytest.mark.parametrize("dt", ["c128", "c64"])
@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("n", [10, 11, 13, 14, 16, 17, 18, 19, 21, 22, 23, 25])
def test_layer_tiles(dt, weighted, n):
    """Every tile size and number of passes, and the cache policies (32 MiB of states from 21
    qubits on): the fused layer and its adjoint against the phase and the gates one by one,
    on a graph of up to 64 edges with repeated ones.  Tolerances: 3 n + 2 roundings per
    amplitude of size <= 1 (2^-53, 2^-24), and for the sums the existing relative ones."""
    from iqs_amd import gates as Gt
    r = np.random.default_rng(n)
    pairs = [tuple(int(v) for v in r.choice(n, 2, replace=False)) for _ in range(min(64, 3 * n))]
    pairs[-1] = pairs[0]
    edges = [(u, v, float(r.uniform(0.1, 2.0)) if weighted else 1.0) for u, v in pairs]
    gamma, beta = 0.37, 0.91
    psi, lam = _state(n, dt, 51), _state(n, dt, 52)
    X = np.array([[0, 1], [1, 0]])
    a, b = _gpu(psi, dt), _gpu(psi, dt)
    a.qaoa_layer(edges, gamma, Gt.rx(2 * beta))
    b.qaoa_phase(edges, gamma)
    for q in range(n):
        b.apply_1q(q, Gt.rx(2 * beta))
    assert a.maxabsdiff(b) < TOL[dt]
    la, lb = _gpu(lam, dt), _gpu(lam, dt)
    b.copy_from(a)
    dg, db = a.qaoa_layer_adjoint(la, edges, gamma, Gt.rx(-2 * beta), X)
    db1 = sum(b.adjoint_1q(lb, q, Gt.rx(-2 * beta), X) for q in range(n))
    dg1 = b.qaoa_phase_adjoint(lb, edges, gamma)
    tol = 1e-11 if dt == "c128" else 2e-5
    assert abs(db - db1) < tol * max(1, abs(db1)) and abs(dg - dg1) < tol * max(1, abs(dg1))
    assert a.maxabsdiff(b) < TOL[dt] and la.maxabsdiff(lb) < TOL[dt]


@pytest.mark.parametrize("dt,n", [(dt, n) for dt in ("c128", "c64") for n in (10, 11, 12, 13, 16, 17, 18, 19, 21, 22, 24, 25)]
                         + [("c64", 26), ("c64", 29)])
def test_general_layer_tiles(dt, n):
    """A general 2x2 and a general generator in every tile size, cache policy and number of passes, with
    and without a weighted phase, and the generator X with a general inverse: against the phase and the
    gates one by one.  Tolerances: 4 n + 2 roundings per amplitude of size <= 1, and for the sums the
    relative ones above."""
    r = np.random.default_rng(n)
    pairs = [tuple(int(v) for v in r.choice(n, 2, replace=False)) for _ in range(min(64, 2 * n))]
    edges = [(u, v, float(r.uniform(0.1, 2.0))) for u, v in pairs]
    gamma, u = 0.37, _unitary(3 * n)
    uinv = u.conj().T
    a, b = StateVector(n, dt), StateVector(n, dt)

    def start(sv, angle):  # a generic state made on the GPU (29 qubits are 4 GiB)
        sv.init_uniform(2.0 ** (-n / 2))
        sv.qaoa_phase(edges, angle)
        for q in range(n):
            sv.apply_1q(q, _unitary(7 * n + q))

    def gates(sv, m):
        for q in range(n):
            sv.apply_1q(q, m)

    start(a, 0.9)
    b.copy_from(a)
    a.apply_1q_all(u)
    gates(b, u)
    assert a.maxabsdiff(b) < TOL[dt]
    a.qaoa_layer(edges, gamma, u)
    b.qaoa_phase(edges, gamma)
    gates(b, u)
    assert a.maxabsdiff(b) < TOL[dt]
    if n > 25:
        return  # the adjoint's tiles are those of 25 qubits
    X = np.array([[0, 1], [1, 0]], dtype=complex)
    G = np.array([[0.3, 1.2 - 0.4j], [1.2 + 0.4j, -0.7]])
    tol = 1e-11 if dt == "c128" else 2e-5
    la, lb = StateVector(n, dt), StateVector(n, dt)
    start(la, 0.2)
    lb.copy_from(la)
    for gen in (G, X):
        b.copy_from(a)
        lb.copy_from(la)
        got = a.adjoint_1q_all(la, uinv, gen)
        want = sum(b.adjoint_1q(lb, q, uinv, gen) for q in range(n))
        assert abs(got - want) < tol * max(1, abs(want))
        assert a.maxabsdiff(b) < TOL[dt] and la.maxabsdiff(lb) < TOL[dt]
    dg, dm = a.qaoa_layer_adjoint(la, edges, gamma, uinv, G)
    dm1 = sum(b.adjoint_1q(lb, q, uinv, G) for q in range(n))
    dg1 = b.qaoa_phase_adjoint(lb, edges, gamma)
    assert abs(dg - dg1) < tol * max(1, abs(dg1)) and abs(dm - dm1) < tol * max(1, abs(dm1))
    assert a.maxabsdiff(b) < TOL[dt] and la.maxabsdiff(lb) < TOL[dt]


@pytest.mark.parametrize("dt", ["c128", "c64"])
@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("n,p", [(10, 20), (13, 20), (18, 20), (10, 300)])
def test_qaoa_circuit_in_one_call(dt, weighted, n, p):
    """qaoa_run and qaoa_gradient against a loop of the layer calls: more sums than one list of runs
    holds (20 layers), and more results than the first buffer has room for (300 layers of 10 qubits).
    The layers are the same kernels, so the states are the same bits; sums that were taken together
    differ by the order of at most 2^8 partials (2^8 roundings of 2^-53 of sums of magnitude up to
    the cost, 2 n)."""
    from iqs_amd import gates as Gt
    edges = _graph(n, 5, weighted)
    r = np.random.default_rng(p)
    gammas, betas = r.uniform(0, np.pi, p), r.uniform(0, np.pi, p)
    X = np.array([[0, 1], [1, 0]])
    a, la, b, lb = (StateVector(n, dt) for _ in range(4))
    a.qaoa_run(edges, gammas, betas)
    b.init_uniform(1.0 / np.sqrt(float(1 << n)))
    for g, t in zip(gammas, betas):
        b.qaoa_layer(edges, g, Gt.rx(2 * t))
    assert a.maxabsdiff(b) == 0.0
    cost, dg, db = a.qaoa_gradient(la, edges, gammas, betas)
    want = b.qaoa_cost_apply(lb, edges)
    tol = 2.0 ** 8 * 2.0 ** -53 * 2 * n
    assert abs(cost - want) < tol
    for l in reversed(range(p)):
        wg, wb = b.qaoa_layer_adjoint(lb, edges, gammas[l], Gt.rx(-2 * betas[l]), X)
        assert abs(dg[l] - wg) < 2 * tol and abs(db[l] - wb) < 2 * tol * n
    assert a.maxabsdiff(b) == 0.0 and la.maxabsdiff(lb) == 0.0
