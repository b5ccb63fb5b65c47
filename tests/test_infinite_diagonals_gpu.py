"""Diagonals with an infinite entry leave the amplitudes that the entry does not
multiply as they are, fused with other diagonals or not."""
import numpy as np
import pytest

from qiskit_aer_amd import QubitVector

pytestmark = pytest.mark.gpu


def state(n, precision, pivot, member, entry):
    """U3 on the qubits of a tile, then phases of one control, which fuse, and a
    diagonal on a qubit outside the tile."""
    rng = np.random.default_rng(n)
    e = QubitVector(n, precision)
    e.initialize()
    u = [np.linalg.qr(rng.standard_normal((2, 2)) + 1j * rng.standard_normal((2, 2)))[0] for _ in range(2 * n)]
    for q in range(n):
        e.apply_matrix([q], u[q])
    e.synchronize()
    for q in range(8):
        e.apply_matrix([q], u[n + q])
    for q in range(pivot):
        e.apply_mcphase([pivot, q], entry if q == member else 1j)
    e.apply_diagonal_matrix([n - 1], [1.0, entry])
    return e.copy_to_vector()


@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("n", [13, 17, 22])
def test_infinite_entries(n, precision):
    print(f"case: infinite diagonal n={n} {precision}", flush=True)
    i = np.arange(1 << n)
    for pivot, member in [(2, 0), (2, 1), (5, 4), (7, 2), (7, 6), (10, 0), (10, 4), (10, 8), (11, 3), (11, 10)]:
        got, want = state(n, precision, pivot, member, np.inf), state(n, precision, pivot, member, 0.5)
        keep = (((i >> pivot) & (i >> member) & 1) | (i >> (n - 1))) == 0
        assert np.all(np.isfinite(got[keep])), (pivot, member)
        # the same operations in maybe another order: a few roundings of each amplitude
        assert np.max(np.abs(got[keep] - want[keep])) < (1e-15 if precision == "double" else 1e-6), (pivot, member)
        assert not np.any(np.isfinite(got[~keep])), (pivot, member)
