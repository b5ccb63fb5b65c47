"""The packed form of a circuit (no device needed): what callers may pass for
qubits, parameters and matrices."""
import numpy as np
import pytest

from qiskit_aer_amd import Circuit, Op
from qiskit_aer_amd import _lib as L


def qubits_of(arr, i):
    return [arr[i].qubits[k] for k in range(arr[i].num_qubits)]


@pytest.mark.parametrize("two", [2.0, np.float64(2.0), np.int32(2), np.uint8(2), "2"])
def test_qubits_that_numpy_converts(two):
    """pauli, measure, reset and barrier keep the qubits as they are given."""
    c = Circuit(4)
    c.gate("h", [0])
    c.pauli("XX", [0.0, two])
    c.measure([two, True], [0, 1])
    c.reset([1.0, 3.0])
    c.barrier(two, 1)
    c.gate("u3", [3], [0.1, 0.2, 0.3])
    arr, keep = c.pack()
    assert [qubits_of(arr, i) for i in range(6)] == [[0], [0, 2], [2, 1], [1, 3], [2, 1], [3]]
    assert [arr[5].params[k] for k in range(3)] == [0.1, 0.2, 0.3]
    assert arr[1].string_param == b"XX"
    del keep


def test_params_that_numpy_converts():
    c = Circuit(2)
    c.ops = [Op(L.OP_GATE, "rx", (0,), ("0.5",)), Op(L.OP_GATE, "cu", (0, 1), (np.array(0.25), 1, np.float32(2), 3.0))]
    arr, keep = c.pack()
    assert arr[0].params[0] == 0.5
    assert [arr[1].params[k] for k in range(4)] == [0.25, 1.0, 2.0, 3.0]
    del keep


def test_negative_qubits_are_refused():
    c = Circuit(2)
    c.pauli("X", [-1])
    with pytest.raises(OverflowError):
        c.pack()


@pytest.mark.parametrize("shape", [(2, 2), (4, 4), (2, 8)])
def test_square_matrices_are_refused(shape):
    """An op's matrix is a vector; the words of a square array could be in
    either order."""
    c = Circuit(2)
    c.ops = [Op(L.OP_MATRIX, "unitary", (0, 1), matrix=np.zeros(shape, dtype=complex).T.copy().T)]
    with pytest.raises(ValueError):
        c.pack()


@pytest.mark.parametrize("values", [np.arange(8.0)[::-2], np.arange(8.0)[::2].astype(np.complex64),
                                    (np.arange(4.0) + 1j).reshape(1, 4), np.array(3.0 + 4.0j)])
def test_vectors_of_any_stride_and_type(values):
    c = Circuit(2)
    c.ops = [Op(L.OP_DIAGONAL, "diagonal", (0, 1), matrix=values)]
    arr, keep = c.pack()
    flat = values.reshape(-1)
    assert arr[0].num_params == flat.size
    got = [complex(arr[0].params[2 * k], arr[0].params[2 * k + 1]) for k in range(flat.size)]
    assert got == [complex(v) for v in flat]
    del keep
