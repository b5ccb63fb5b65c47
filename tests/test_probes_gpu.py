"""Saved Pauli values in every form the planner gives them: runs of probes in
register passes, probes on the LDS tile, sweeps of wide strings, more than one
batch of either, and the same inside batched circuits of several sizes."""
import numpy as np
import pytest

from oracle import pyoracle as O
from tests import dense as D

pytestmark = pytest.mark.gpu


def pauli_value(psi, label):
    n = len(label)
    x = sum(1 << (n - 1 - i) for i, p in enumerate(label) if p in "XY")
    z = [n - 1 - i for i, p in enumerate(label) if p in "YZ"]
    i = np.arange(psi.size)
    parity = np.zeros_like(i)
    for q in z:
        parity ^= i >> q
    return float(np.real(1j ** label.count("Y") * np.sum(np.conj(psi[i ^ x]) * psi * (1 - 2.0 * (parity & 1)))))


def strings(n, count, rng):
    out = ["".join("IXYZ"[k] for k in rng.integers(0, 4, n)) for _ in range(count)]
    for q in range(n):  # and local ones, which share tile passes
        for p in "XYZ":
            out.append("I" * (n - 1 - q) + p + "I" * q)
    return out


@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("n,tile_bits", [(5, 0), (11, 0), (12, 0), (13, 0), (15, 0), (17, 0), (12, 6), (14, 9)])
def test_probes_match_dense(n, tile_bits, precision):
    from qiskit_aer_amd import QubitVector
    print(f"case: probes n={n} tile={tile_bits} {precision}", flush=True)
    rng = np.random.default_rng(n)
    psi = D.random_state(n, rng)
    if precision == "single":
        psi = psi.astype(np.complex64).astype(np.complex128)
    e = QubitVector(n, precision)
    if tile_bits:
        e.set_tile_bits(tile_bits, 2)
    e.initialize_from_vector(psi)
    labels = strings(n, 150, rng)
    got = e.expval_pauli_multi(list(range(n)), labels)
    # FP64 products and sums of at most 2^17 terms that add up to 1 in magnitude
    assert np.max(np.abs(got - [pauli_value(psi, lab) for lab in labels])) < 1e-13
    # a phase with both parts: Re(phase <P>) of Hermitian P
    some = labels[:6] + labels[-4:]
    slots = [e.save_expval_pauli(list(range(n)), lab, 0.6 - 0.8j) for lab in some]
    vals = e.saved_expvals()
    want = [0.6 * pauli_value(psi, lab) for lab in some]
    assert np.max(np.abs(vals[slots] - want)) < 1e-13


@pytest.mark.parametrize("precision", ["double", "single"])
def test_batched_circuits_with_many_strings(precision):
    from qiskit_aer_amd import circuits
    from qiskit_aer_amd.batch import batch_pauli_expval
    sizes = [16, 3, 12, 14, 14, 11, 14, 12, 1]
    print(f"case: batch of {sizes} with 70 strings {precision}", flush=True)
    rng = np.random.default_rng(3)
    cs, hs, want = [], [], []
    for k, n in enumerate(sizes):
        if n > 1:
            c, _ = circuits.hea(n, 1 + k % 4, 20 + k)
        else:
            c = circuits.Circuit(1)
            c.gate("h", [0])
        if k == 4:  # a SWAP layer, and a gate that needs the LDS tile
            for q in range(n // 2):
                c.gate("swap", [q, n - 1 - q])
            c.unitary(D.random_unitary(8, rng), [0, 5, 9])
        labels = strings(n, 70, rng)
        h = list(zip(labels, rng.standard_normal(len(labels))))
        _, psi, _ = O.run_circuit(c, shots=0, seed=0, fusion=False)
        cs.append(c)
        hs.append(h)
        want.append(sum(w * pauli_value(psi, lab) for lab, w in h))
    got, _ = batch_pauli_expval(cs, hs, precision)
    assert np.max(np.abs(got - want)) < (1e-10 if precision == "double" else 1e-4)
