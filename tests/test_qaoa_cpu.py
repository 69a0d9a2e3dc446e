"""MaxCutQaoa's arguments, without a GPU: the engine calls of a 10-qubit problem (the size from which
whole circuits are one call) recorded by a stand-in for the state vector."""
import numpy as np
import pytest

from iqs_amd.qaoa import LAYER_MIN_QUBITS, MaxCutQaoa


class Recorder:
    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def call(*args):
            # The ctypes call takes doubles: the same conversion.
            if name in ("qaoa_run", "qaoa_gradient"):
                args = args[:-2] + tuple(np.ascontiguousarray(a, dtype=np.float64).reshape(-1).tolist() for a in args[-2:])
            self.calls.append((name, args))
            return (0.0, np.zeros(1), np.zeros(1)) if name == "qaoa_gradient" else None

        return call


def _problem(edges=None):
    p = MaxCutQaoa(LAYER_MIN_QUBITS, edges or [(0, 1, 1.0), (1, 2, 1.0)])
    p._psi, p._lam = Recorder(), Recorder()
    return p


class Scalar:
    """A number that only converts to float, one by one (as tensors on a device do)."""

    def __init__(self, v):
        self.v = v

    def __rmul__(self, o):
        return Scalar(o * self.v)

    def __float__(self):
        return float(self.v)


@pytest.mark.parametrize("kind", ["list", "generator", "array", "float32", "scalars", "tensor"])
def test_angles_of_any_type(kind):
    g, b = [0.5, 0.25], [1.0, 2.0]
    make = {"list": list, "generator": iter, "array": np.array, "float32": lambda v: np.array(v, dtype=np.float32),
            "scalars": lambda v: [Scalar(x) for x in v]}.get(kind)
    if kind == "tensor":
        torch = pytest.importorskip("torch")
        make = lambda v: torch.tensor(v, requires_grad=True)  # noqa: E731
    p = _problem()
    p.forward_state(make(g), make(b))
    assert p._psi.calls == [("qaoa_run", (p.edges, g, b))]
    if kind != "generator":
        p._psi.calls.clear()
        p.adjoint_from_final(make(g), make(b))
        assert p._psi.calls == [("qaoa_gradient", (p._lam, p.edges, g, b))]


def test_lengths_and_refused_angles():
    p = _problem()
    p.forward_state([0.5, 0.25, 9.0], [1.0, 2.0])  # the shorter list counts
    assert p._psi.calls.pop() == ("qaoa_run", (p.edges, [0.5, 0.25], [1.0, 2.0]))
    p.adjoint_from_final([0.5], [1.0, 2.0])
    assert p._psi.calls.pop() == ("qaoa_gradient", (p._lam, p.edges, [0.5], [1.0]))
    with pytest.raises(IndexError):
        p.adjoint_from_final([0.5, 0.25], [1.0])
    for bad in ([[0.5, 0.25]], ["0.5"], [1j]):
        with pytest.raises(TypeError):
            p.forward_state(bad if bad != [[0.5, 0.25]] else np.array(bad), [1.0])
    assert p._psi.calls == []


def test_no_layers_on_any_graph():
    p = _problem([(i % 9, 9, 1.0) for i in range(70)])  # more edges than a phase takes
    p.forward_state([], [])
    assert p._psi.calls == [("init_uniform", (1.0 / 32.0,))]
