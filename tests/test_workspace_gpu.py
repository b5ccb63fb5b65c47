"""Handles that follow one another share their stream and buffers: results do
not depend on what an earlier handle of another size, precision or use left,
nor on several threads creating and ending handles at once."""
import threading

import numpy as np
import pytest

from tests import dense as D

pytestmark = pytest.mark.gpu


def check(n, precision, seed):
    from qiskit_aer_amd import QubitVector
    psi = D.random_state(n, np.random.default_rng(seed))
    e = QubitVector(n, precision)
    e.initialize_from_vector(psi)
    u = D.random_unitary(2, np.random.default_rng(seed + 1))
    e.apply_matrix([n - 1], u)
    want = D.apply(psi, u, [n - 1])
    tol = 1e-13 if precision == "double" else 1e-6
    ok = np.max(np.abs(e.copy_to_vector() - want)) < tol
    p = np.abs(want) ** 2
    ok &= abs(e.norm() - p.sum()) < 10 * tol
    ok &= np.max(np.abs(e.probabilities([0]) - [p[0::2].sum(), p[1::2].sum()])) < 10 * tol
    draws = np.random.default_rng(seed).random(50)
    got = e.sample_measure(draws).astype(np.int64)
    cdf = np.cumsum(p)
    ok &= bool(np.all(draws < cdf[got] + 10 * tol))
    e.close()
    return bool(ok)


def test_sizes_and_precisions_in_turn():
    print("case: handles in turn", flush=True)
    for k, (n, precision) in enumerate([(5, "double"), (5, "single"), (20, "double"), (5, "double"), (23, "double"),
                                        (20, "single"), (3, "double"), (20, "double"), (1, "single")]):
        assert check(n, precision, k), (n, precision)


def test_many_alive_at_once():
    from qiskit_aer_amd import QubitVector
    print("case: more handles alive than the pool keeps", flush=True)
    for _ in range(2):
        qs = [QubitVector(4 + k) for k in range(7)]
        for q in qs:
            q.initialize()
            q.apply_mcx([0])
        for q in qs:
            v = q.copy_to_vector()
            assert v[1] == 1 and np.count_nonzero(v) == 1
        for q in qs:
            q.close()


def test_threads():
    print("case: handles from 4 threads", flush=True)
    bad = []

    def work(t):
        for k in range(6):
            n = 3 + (5 * t + k) % 12
            if not check(n, "double" if k % 2 else "single", 100 * t + k):
                bad.append((t, k, n))

    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
