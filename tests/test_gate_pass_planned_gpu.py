"""Gate passes are what the circuits below run in, where the planner takes them,
and are not where it does not: the counts of the handle, with the values."""
import numpy as np
import pytest

from oracle import pyoracle as O
from qiskit_aer_amd import QubitVector, circuits
from tests import dense as D
from tests.test_gate_pass_gpu import mixture, pauli_value, wide_mixture

pytestmark = pytest.mark.gpu


def run(c, n, precision, width=0):
    e = QubitVector(n, precision)
    e.set_block_fusion(width)
    e.initialize()
    e.apply_ops(c)
    e.synchronize()
    _, want, _ = O.run_circuit(c, shots=0, seed=0, fusion=False)
    # a gate rounds the state by at most 4 (16 for 8x8 gates) parts of the norm
    bound = len(c.ops) * 16 * (2.0**-53 if precision == "double" else 2.0**-24)
    assert np.linalg.norm(e.copy_to_vector() - want) < bound
    return e.gate_pass_stats()


@pytest.mark.parametrize("precision,n,taken", [("double", 20, False), ("double", 21, True), ("single", 12, True),
                                               ("single", 17, True)])
def test_mixed_gates(precision, n, taken):
    print(f"case: planned gate passes {precision} n={n}", flush=True)
    for c in (mixture(n, 51, 120), wide_mixture(n, 52, 40)):
        passes, _ = run(c, n, precision)
        assert (passes > 0) == taken


@pytest.mark.parametrize("precision,n", [("double", 21), ("single", 13)])
def test_cx_chains_with_4x4_gates(precision, n):
    """CX and X on every ordered pair of a tile's qubits between gates that force
    layout changes."""
    print(f"case: planned CX in layout changes {precision} n={n}", flush=True)
    rng = np.random.default_rng(n + 60)
    c = circuits.Circuit(n)
    pairs = [(a, b) for a in range(12) for b in range(12) if a != b]
    for k, i in enumerate(rng.permutation(len(pairs))):
        a, b = pairs[int(i)]
        c.gate("cx", [a, b])
        if k % 5 == 0:
            c.gate("x", [int(rng.integers(12))])
        if k % 7 == 0 or 40 < k < 60:
            c.unitary(D.random_unitary(4, rng), [int(q) for q in rng.choice(12, 2, replace=False)])
            c.gate("u3", [int(rng.integers(12))], list(rng.uniform(-3, 3, 3)))
    passes, cx = run(c, n, precision)
    assert passes > 0 and cx > 10


@pytest.mark.parametrize("precision,n", [("double", 21), ("single", 13)])
def test_probes(precision, n):
    print(f"case: planned probes {precision} n={n}", flush=True)
    c = mixture(n, 53, 40)
    _, psi, _ = O.run_circuit(c, shots=0, seed=0, fusion=False)
    e = QubitVector(n, precision)
    e.initialize()
    e.apply_ops(c)
    labels = ["I" * (n - 1 - q) + p + "I" * q for q in range(n) for p in "XYZ"]
    slots = [e.save_expval_pauli(list(range(n)), lab, 1.0) for lab in labels]
    got = e.saved_expvals()[slots]
    bound = 1e-12 if precision == "double" else 2 * len(c.ops) * 16 * 2.0**-24
    assert np.max(np.abs(got - [pauli_value(psi, lab) for lab in labels])) < bound
    assert e.gate_pass_stats()[0] > 0


def lean_gates(n, seed):
    """Two layers of 2x2 gates, CX and phases on a window of 12 qubits."""
    rng = np.random.default_rng(seed)
    c = circuits.Circuit(n)
    for layer in range(2):
        for q in range(12):
            c.gate("u3", [n - 1 - q], list(rng.uniform(-3, 3, 3)))
        for q in range(layer, 11, 2):
            c.gate("cx", [n - 1 - q, n - 2 - q])
        for q in range(3):
            c.gate("cp", [n - 1 - q, n - 6 - q], [float(rng.uniform(-3, 3))])
            c.gate("rz", [n - 2 - q], [float(rng.uniform(-3, 3))])
    return c


@pytest.mark.parametrize("precision,n,taken", [("double", 13, False), ("double", 21, False), ("double", 22, True),
                                               ("single", 13, False), ("single", 22, False), ("single", 23, True)])
def test_lean_gates_on_few_tiles(precision, n, taken):
    """With fewer tiles a pass of 2x2 gates, X and phases is a register pass."""
    print(f"case: planned lean gates {precision} n={n}", flush=True)
    passes, _ = run(lean_gates(n, 54), n, precision)
    assert (passes > 0) == taken


def test_lean_passes_beside_others_with_few_tiles():
    """The lean stretch of a circuit runs in register passes, the 4x4 gates in
    gate passes."""
    n = 21
    print("case: planned lean and 4x4 gates", flush=True)
    c = lean_gates(n, 55)
    rng = np.random.default_rng(56)
    for q in range(8):
        c.unitary(D.random_unitary(4, rng), [q, q + 1])
    passes, _ = run(c, n, "double")
    assert passes > 0


@pytest.mark.parametrize("precision,low,passes", [("double", True, 1), ("double", False, 0), ("single", True, 0),
                                                  ("single", False, 0)])
def test_shallow_lean_segments(precision, low, passes):
    """12 gates on 12 qubits: in complex128 one gate pass instead of two register
    passes where the tile's low bits are among them, otherwise no fewer passes."""
    n = 23
    print(f"case: planned shallow gates {precision} low={low}", flush=True)
    rng = np.random.default_rng(57)
    c = circuits.Circuit(n)
    for q in range(12):
        c.gate("u3", [q if low else n - 1 - q], list(rng.uniform(-3, 3, 3)))
    assert run(c, n, precision)[0] == passes
