"""Draws from a state with a NaN amplitude: those below the sums that hold it
are what they are without it, the others end on the last amplitude."""
import numpy as np
import pytest

from qiskit_aer_amd import QubitVector
from tests import dense as D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("n,index_size", [(3, 10), (10, 10), (12, 10), (14, 10), (16, 10), (18, 8)])
def test_draws_before_a_nan(n, index_size, precision):
    print(f"case: draws before a NaN n={n} {precision}", flush=True)
    rng = np.random.default_rng(n)
    psi = D.random_state(n, rng)
    if precision == "single":
        psi = psi.astype(np.complex64).astype(np.complex128)
    total = np.cumsum(np.abs(psi) ** 2)
    at = 3 << (n - 2)  # the NaN: at the first amplitude of an index block
    draws = np.concatenate([rng.random(500) * total[at - 1] * (1 - 1e-9), [total[at - 1] + 1e-6, 0.999]])
    bad = psi.copy()
    bad[at] = np.nan
    e = QubitVector(n, precision)
    e.set_sample_measure_index_size(index_size)
    e.initialize_from_vector(bad)
    got = e.sample_measure(draws).astype(np.int64)
    e.initialize_from_vector(psi)
    want = e.sample_measure(draws).astype(np.int64)
    assert np.array_equal(got[:500], want[:500])
    assert np.all(got[500:] == (1 << n) - 1)
