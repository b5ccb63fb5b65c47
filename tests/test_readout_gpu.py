"""Readout kernels at the edges of their ranges: marginal probabilities over
lane and higher qubits, long rows of partial sums, and the sampling index with
one run per block, several, and more than one LDS chunk of either."""
import numpy as np
import pytest

from tests import dense as D

pytestmark = pytest.mark.gpu


def loaded(n, precision, seed):
    from qiskit_aer_amd import QubitVector
    psi = D.random_state(n, np.random.default_rng(seed))
    if precision == "single":
        psi = psi.astype(np.complex64).astype(np.complex128)
    e = QubitVector(n, precision)
    e.initialize_from_vector(psi)
    return e, np.abs(psi) ** 2


@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("n", [1, 4, 6, 7, 13, 18])
def test_marginals_of_any_qubits(n, precision):
    print(f"case: marginals n={n} {precision}", flush=True)
    e, p = loaded(n, precision, n)
    rng = np.random.default_rng(n + 1)
    sets = [rng.permutation(n)[:k] for k in sorted({1, min(2, n), n // 2, n - 1, n}) if k > 0]
    sets += [np.arange(n)[::-1]]
    t = p.reshape([2] * n)
    for qs in sets:
        axes = [n - 1 - int(q) for q in reversed(qs)]
        rest = tuple(a for a in range(n) if a not in axes)
        want = np.transpose(t, axes + list(rest)).reshape(1 << len(qs), -1).sum(axis=1)
        # up to 2^18 non-negative terms, each sum rounded to one part in 2^53
        assert np.max(np.abs(e.probabilities(list(qs)) - want)) < 1e-14, list(qs)


@pytest.mark.parametrize("n,index_size", [(3, 10), (10, 10), (11, 10), (14, 13), (15, 3), (23, 1), (20, 10)])
def test_draws_fall_in_their_own_interval(n, index_size):
    print(f"case: draws n={n} index size {index_size}", flush=True)
    e, p = loaded(n, "double", n)
    e.set_sample_measure_index_size(index_size)
    total = np.cumsum(p)
    draws = np.concatenate([np.random.default_rng(5).random(700), [0.0, total[-1] * (1 - 1e-9), 1.0 + 1e-9]])
    got = e.sample_measure(draws).astype(np.int64)
    assert got[-1] == (1 << n) - 1
    # cumulative sums of at most 2^23 terms differ by the order of addition
    # alone, less than 2^23 * 2^-53 of a total of 1
    below = np.where(got > 0, total[np.maximum(got - 1, 0)], 0.0)
    assert np.all(below[:-1] <= draws[:-1] + 1e-9)
    assert np.all(draws[:-1] < total[got[:-1]] + 1e-9)
    exact = np.searchsorted(total, draws[:-1], side="right")
    assert np.mean(got[:-1] != exact) < 0.01


@pytest.mark.parametrize("n", [3, 12, 16, 22])
def test_norm_and_pauli_rows(n):
    """Rows of 1 to 4096 partials (norm, one Pauli string) and one partial per
    tile of saved values."""
    print(f"case: rows n={n}", flush=True)
    e, p = loaded(n, "double", n)
    assert abs(e.norm() - p.sum()) < 1e-13
    z = 1.0 - 2.0 * ((np.arange(1 << n) >> (n - 1)) & 1)
    want = float((p * z).sum())
    assert abs(e.expval_pauli([n - 1], "Z") - want) < 1e-13
    got = e.expval_pauli_multi([0, n - 1], ["ZI", "IZ", "XX"])
    assert abs(got[0] - want) < 1e-13
    psi = e.copy_to_vector()
    flip = np.arange(1 << n) ^ (1 | 1 << (n - 1))
    assert abs(got[2] - float(np.real(np.vdot(psi, psi[flip])))) < 1e-13
