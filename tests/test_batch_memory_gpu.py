"""Batched circuits with more Pauli terms than one pass holds: the values, and
that the device memory of a call does not grow with terms times tiles."""
import threading

import numpy as np
import pytest

from qiskit_aer_amd import circuits
from qiskit_aer_amd.batch import batch_pauli_expval
from qiskit_aer_amd.qubitvector import device_memory

pytestmark = pytest.mark.gpu


def terms_of(n, count, seed, letters):
    rng = np.random.default_rng(seed)
    rows = rng.choice(list(letters), size=(count, n))
    return [("".join(r), float(c)) for r, c in zip(rows, rng.standard_normal(count))]


@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("letters", ["IZ", "IXYZ", "IIIIIIIIIX"])
def test_more_terms_than_a_pass_holds(precision, letters):
    """Diagonal terms fill register passes, terms with X on all qubits sweeps,
    few X tile passes with others left for later ones; 256 terms a pass."""
    print(f"case: many terms {precision} {letters}", flush=True)
    sizes, counts = [11, 12, 13, 14, 13], [700, 300, 257, 600, 256]
    cs = [circuits.hea(n, 2, 40 + n)[0] for n in sizes]
    hs = [terms_of(n, k, 60 + i, letters) for i, (n, k) in enumerate(zip(sizes, counts))]
    got, _ = batch_pauli_expval(cs, hs, precision, "batch")
    want, _ = batch_pauli_expval(cs, hs, precision, "sequential")
    # each value is within a few roundings of the state's (2^-53, 2^-24) of the
    # other's, and 700 normal weights add up to less than 700 in magnitude
    assert np.max(np.abs(got - want)) < 700 * (1e-14 if precision == "double" else 2e-6)


def test_memory_of_many_terms():
    """20 000 terms on 2^10 tiles: 160 MiB if every term kept a partial per tile;
    the state is 32 MiB."""
    print("case: memory of a batch with many terms", flush=True)
    n, count = 21, 20000
    c, _ = circuits.hea(n, 1, 3)
    h = terms_of(n, count, 5, "IZ")
    batch_pauli_expval([c], [h[:300]])  # code objects, the first buffers
    out = []
    before = device_memory()[0]
    worker = threading.Thread(target=lambda: out.append(batch_pauli_expval([c], [h])[0][0]))
    worker.start()
    least = before
    while worker.is_alive():
        least = min(least, device_memory()[0])
    worker.join()
    part = sum(batch_pauli_expval([c], [h[k:k + 5000]])[0][0] for k in range(0, count, 5000))
    assert abs(out[0] - part) < 1e-9
    assert before - least < (100 << 20)
