"""Gate passes (tiles of 2^12 amplitudes; complex128 from 21 qubits on): every
op they run, on qubits inside and outside the tile, next to ops they leave to
the other passes, against the oracle; and the same gates just below 21 qubits."""
import numpy as np
import pytest

from oracle import pyoracle as O
from qiskit_aer_amd import QubitVector, circuits
from tests import dense as D

pytestmark = pytest.mark.gpu


def run_both(c, n, width=0, state=None):
    e = QubitVector(n)
    e.set_block_fusion(width)
    e.initialize()
    e.apply_ops(c)
    _, want, _ = O.run_circuit(c, shots=0, seed=0, fusion=False)
    return float(np.max(np.abs(e.copy_to_vector() - want)))


def mixture(n, seed, count):
    """Gates of every kind, most of them on a window of nearby qubits so that a
    pass holds many."""
    rng = np.random.default_rng(seed)
    c = circuits.Circuit(n)
    for q in range(n):
        c.gate("h", [q])
    for _ in range(count):
        lo = int(rng.integers(0, n - 5)) if rng.random() < 0.8 else 0
        hi = lo + 6 if lo or rng.random() < 0.5 else n
        q = [int(x) for x in rng.choice(np.arange(lo, min(hi, n)), 3, replace=False)]
        t = list(rng.uniform(-3, 3, 3))
        k = int(rng.integers(16))
        if k < 4:
            c.gate("u3", q[:1], t)
        elif k < 7:
            c.gate("cx", q[:2])
        elif k == 7:
            c.unitary(D.random_unitary(4, rng), q[:2])
        elif k == 8:
            c.gate("rz", q[:1], t[:1])
        elif k == 9:
            c.gate("cp", q[:2], t[:1])
        elif k == 10:
            c.gate("ccx", q)
        elif k == 11:
            c.gate("cu3", q[:2], t)
        elif k == 12:
            c.gate("cy", q[:2])
        elif k == 13:
            c.gate("x", q[:1])
        elif k == 14:
            c.gate("mcp", q, t[:1])
        else:
            c.gate("swap", q[:2]) if rng.random() < 0.3 else c.gate("y", q[:1])
    return c


@pytest.mark.parametrize("n,seed", [(20, 1), (21, 2), (21, 3), (22, 4)])
def test_mixture_matches_oracle(n, seed):
    print(f"case: gate pass mixture n={n} seed={seed}", flush=True)
    # 300 gates, each rounding amplitudes of at most 1 to a few 2^-53
    assert run_both(mixture(n, seed, 300), n) < 1e-12


@pytest.mark.parametrize("width", [0, 2, 3])
def test_brickwork_fused_and_not(width):
    n = 21
    print(f"case: gate pass brickwork n={n} width={width}", flush=True)
    assert run_both(circuits.brickwork_u3_cx(n, 12, 5, measure=False), n, width) < 1e-12


def test_qft_ladders():
    """Fused diagonals: lane tables staged in LDS, and beyond eight of them read
    from memory."""
    n = 22
    print(f"case: gate pass qft n={n}", flush=True)
    c = circuits.qft(n)
    assert run_both(c, n) < 1e-12


def test_gradients_use_them():
    """The forward sweep of the adjoint method holds no probes."""
    from qiskit_aer_amd.adjoint import AdjointEstimator
    from bench import ry_rz_cz_ansatz, tfim
    n = 20  # 21 with the flag qubit
    print(f"case: gate pass gradients n={n}", flush=True)
    c, idx, npar = ry_rz_cz_ansatz(n, 3)
    est = AdjointEstimator(c, idx, npar, tfim(n))
    rows = np.random.default_rng(2).uniform(-3, 3, size=(2, npar))
    e, g = est.energy_and_gradient(rows)
    assert np.max(np.abs(e - est.energy_one_by_one(rows))) < 1e-11
    which = [0, npar // 2, npar - 1]
    assert np.max(np.abs(est.parameter_shift(rows[:1], which)[0] - g[0, which])) < 1e-9


@pytest.mark.parametrize("width", [0, 2, 3])
@pytest.mark.parametrize("n,seed", [(12, 5), (13, 6), (17, 7), (20, 8)])
def test_complex64(n, seed, width):
    """2x2 and 4x4 gates on the matrix cores, from one tile (12 qubits) on."""
    print(f"case: complex64 gate pass n={n} seed={seed} width={width}", flush=True)
    c = mixture(n, seed, 200)
    e = QubitVector(n, "single")
    e.set_block_fusion(width)
    e.initialize()
    e.apply_ops(c)
    _, want, _ = O.run_circuit(c, shots=0, seed=0, fusion=False)
    # a gate is unitary and rounds each amplitude to a few 2^-24 of its group's
    # norm: at most 4 * 2^-24 a gate in the norm of the state
    assert np.linalg.norm(e.copy_to_vector() - want) < (200 + n) * 4 * 2.0**-24


def test_complex64_pairs():
    """A 4x4 gate on every ordered pair of a tile's qubits, then all of a register."""
    n = 13
    rng = np.random.default_rng(9)
    print("case: complex64 4x4 gates on every pair", flush=True)
    c = circuits.Circuit(n)
    for a in range(n):
        for b in range(n):
            if a != b:
                c.unitary(D.random_unitary(4, rng), [a, b])
    e = QubitVector(n, "single")
    e.initialize()
    e.apply_ops(c)
    _, want, _ = O.run_circuit(c, shots=0, seed=0, fusion=False)
    assert np.linalg.norm(e.copy_to_vector() - want) < n * (n - 1) * 8 * 2.0**-24


def wide_mixture(n, seed, count):
    """What needs three register bits, or none: 8x8 gates on every order of their
    qubits, (controlled) swaps, diagonals of one to nine qubits with and without
    controls, between 2x2 gates."""
    rng = np.random.default_rng(seed)
    c = circuits.Circuit(n)
    for q in range(n):
        c.gate("h", [q])
    for _ in range(count):
        lo = int(rng.integers(0, n - 8)) if rng.random() < 0.7 else 0
        q = [int(x) for x in rng.choice(np.arange(lo, n if lo == 0 else lo + 9), 9, replace=False)]
        k = int(rng.integers(9))
        if k < 2:
            c.unitary(D.random_unitary(8, rng), q[:3])
        elif k == 2:
            c.gate("swap", q[:2])
        elif k == 3:
            c.gate("cswap", q[:3])
        elif k == 4:
            w = int(rng.integers(1, 10))
            c.diagonal(np.exp(1j * rng.uniform(-3, 3, 1 << w)), q[:w])
        elif k == 5:
            c.gate("rzz", q[:2], [float(rng.uniform(-3, 3))])
        elif k == 6:
            c.gate("crz", q[:2], [float(rng.uniform(-3, 3))])
        elif k == 7:
            c.gate("cx", q[:2])
        else:
            c.gate("u3", q[:1], list(rng.uniform(-3, 3, 3)))
    return c


@pytest.mark.parametrize("n,seed", [(21, 11), (22, 12)])
def test_wide_ops(n, seed):
    print(f"case: gate pass wide ops n={n} seed={seed}", flush=True)
    assert run_both(wide_mixture(n, seed, 120), n) < 1e-12


@pytest.mark.parametrize("n,seed", [(12, 13), (13, 14), (18, 15)])
def test_wide_ops_complex64(n, seed):
    print(f"case: complex64 gate pass wide ops n={n} seed={seed}", flush=True)
    c = wide_mixture(n, seed, 120)
    e = QubitVector(n, "single")
    e.initialize()
    e.apply_ops(c)
    _, want, _ = O.run_circuit(c, shots=0, seed=0, fusion=False)
    # as above; a component of an 8x8 gate is a sum of 16 rounded products
    assert np.linalg.norm(e.copy_to_vector() - want) < (120 + n) * 16 * 2.0**-24


def pauli_value(psi, label):
    n = len(label)
    x = sum(1 << (n - 1 - i) for i, p in enumerate(label) if p in "XY")
    i = np.arange(psi.size)
    parity = np.zeros_like(i)
    for k, p in enumerate(label):
        if p in "YZ":
            parity ^= i >> (n - 1 - k)
    return float(np.real(1j ** label.count("Y") * np.sum(np.conj(psi[i ^ x]) * psi * (1 - 2.0 * (parity & 1)))))


@pytest.mark.parametrize("precision,n,seed", [("double", 21, 21), ("double", 22, 22), ("single", 12, 23),
                                              ("single", 13, 24), ("single", 16, 25)])
def test_probes_between_gates(precision, n, seed):
    """Saved Pauli values between gates of one queue: X and Y on none to seven
    qubits inside and outside a tile, more of them than a batch holds, 3-qubit
    gates and swaps next to them, and a read-only end."""
    print(f"case: gate pass probes {precision} n={n} seed={seed}", flush=True)
    rng = np.random.default_rng(seed)
    e = QubitVector(n, precision)
    e.initialize()
    want, slots, psi = [], [], None
    prefix = circuits.Circuit(n)
    blocks = [mixture(n, seed, 30), wide_mixture(n, seed + 1, 12), mixture(n, seed + 2, 20)]
    for k, c in enumerate(blocks):
        e.apply_ops(c)
        for op in c.ops:
            prefix.ops.append(op)
        _, psi, _ = O.run_circuit(prefix, shots=0, seed=0, fusion=False)
        for i in range(70 if k == 2 else 8):
            lab = ["I"] * n
            at = rng.permutation(n)
            for q in at[: int(rng.integers(0, 8))]:
                lab[q] = "XY"[int(rng.integers(2))]
            for q in at[8: 8 + int(rng.integers(0, 4))]:
                lab[q] = "Z"
            if i % 2:  # local strings, which share tiles
                q = int(rng.integers(0, n - 1))
                lab = ["I"] * n
                lab[q], lab[q + 1] = "XYZ"[int(rng.integers(3))], "IXYZ"[int(rng.integers(4))]
            lab = "".join(lab)
            slots.append(e.save_expval_pauli(list(range(n)), lab, 1.0))
            want.append(pauli_value(psi, lab))
    got = e.saved_expvals()[slots]
    # FP64 sums; the state before them within 4 (16 for 8x8 gates) roundings of
    # its norm per gate, which a value of a Pauli string doubles
    gates = sum(len(c.ops) for c in blocks)
    bound = 1e-12 if precision == "double" else 2 * gates * 16 * 2.0**-24
    assert np.max(np.abs(got - np.array(want))) < bound
    assert np.linalg.norm(e.copy_to_vector() - psi) < bound


@pytest.mark.parametrize("precision,n", [("double", 21), ("single", 13)])
def test_cx_taken_by_layout_changes(precision, n):
    """CX and X on every ordered pair of a tile's qubits between gates that force
    layout changes: chains of them, more than one layout change takes, before,
    between and after the gates."""
    print(f"case: CX in layout changes {precision} n={n}", flush=True)
    rng = np.random.default_rng(n)
    c = circuits.Circuit(n)
    for _ in range(3):
        for q in range(12):
            c.gate("u3", [q], list(rng.uniform(-3, 3, 3)))
    pairs = [(a, b) for a in range(12) for b in range(12) if a != b]
    for k, i in enumerate(rng.permutation(len(pairs))):
        a, b = pairs[int(i)]
        c.gate("cx", [a, b])
        if k % 5 == 0:
            c.gate("x", [int(rng.integers(12))])
        if k % 7 == 0 or 40 < k < 60:
            c.gate("u3", [int(rng.integers(12))], list(rng.uniform(-3, 3, 3)))
        if k % 11 == 0:
            c.gate("cp", [a, int((b + 1) % 12) if (b + 1) % 12 != a else b], [float(rng.uniform(-3, 3))])
    e = QubitVector(n, precision)
    e.initialize()
    e.apply_ops(c)
    _, want, _ = O.run_circuit(c, shots=0, seed=0, fusion=False)
    bound = 1e-12 if precision == "double" else len(c.ops) * 4 * 2.0**-24
    assert np.linalg.norm(e.copy_to_vector() - want) < bound


def test_replayed_launches_follow_the_probes():
    """Two flushes of one size and pass count whose probes sit in different
    passes: the second does not replay the launches captured for the first."""
    n = 20
    print("case: gate pass probes under replay", flush=True)
    rng = np.random.default_rng(31)
    c = circuits.Circuit(n)
    for lo in (4, 12):  # two passes, a swap and more than a handful of gates in each
        for layer in range(3):
            for q in range(lo, lo + 8):
                c.gate("u3", [q], list(rng.uniform(-3, 3, 3)))
            for q in range(lo + layer % 2, lo + 7, 2):
                c.gate("cx", [q, q + 1])
        c.gate("swap", [lo, lo + 5])
    _, psi, _ = O.run_circuit(c, shots=0, seed=0, fusion=False)

    def label(q):
        return "".join("X" if n - 1 - i == q else "I" for i in range(n))

    e = QubitVector(n, "single")
    for q in (13, 13, 13, 13, 5, 5, 13, 5):
        e.initialize()
        e.apply_ops(c)
        slot = e.save_expval_pauli(list(range(n)), label(q), 1.0)
        got = e.saved_expvals()[slot]
        # 4 roundings of 2^-24 of the norm per gate, doubled by the value
        assert abs(got - pauli_value(psi, label(q))) < 2 * len(c.ops) * 4 * 2.0**-24


@pytest.mark.parametrize("precision,n,rounds", [("double", 21, 10), ("single", 13, 40)])
def test_cx_stay_before_the_probes_they_change(precision, n, rounds):
    """CX, then a run of probes of which a later one sees them, then gates that
    change the layout: the layout change takes no CX past the run."""
    print(f"case: CX before probe runs {precision} n={n}", flush=True)
    rng = np.random.default_rng(n + rounds)
    prefix = circuits.Circuit(n)
    e = QubitVector(n, precision)
    e.initialize()
    want, slots, gates = [], [], 0
    for r in range(rounds):
        c = circuits.Circuit(n)
        if r == 0:
            for q in range(n):
                c.gate("u3", [q], list(rng.uniform(-3, 3, 3)))
        for q in rng.choice(12, 2, replace=False):
            c.gate("u3", [int(q)], list(rng.uniform(-3, 3, 3)))
        a, b, other = (int(x) for x in rng.choice(12, 3, replace=False))
        c.gate("cx", [a, b])
        e.apply_ops(c)
        gates += len(c.ops)
        prefix.ops.extend(c.ops)
        _, psi, _ = O.run_circuit(prefix, shots=0, seed=0, fusion=False)
        for q, p in ((other, "X"), (b, "Z"), (a, "X"), (b, "Y")):
            lab = "".join(p if n - 1 - i == q else "I" for i in range(n))
            slots.append(e.save_expval_pauli(list(range(n)), lab, 1.0))
            want.append(pauli_value(psi, lab))
    got = e.saved_expvals()[slots]
    bound = 1e-12 if precision == "double" else 2 * gates * 4 * 2.0**-24
    assert np.max(np.abs(got - np.array(want))) < bound
