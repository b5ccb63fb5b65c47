"""Device memory that readouts of a handle take beside its state: the buffers
grow to what a call needs and no further."""
import numpy as np
import pytest

from qiskit_aer_amd import QubitVector
from qiskit_aer_amd.qubitvector import device_memory

pytestmark = pytest.mark.gpu

N = 22  # 2^22 doubles are 32 MiB
ROW = 8 << N


def taken(call):
    """Device memory a fresh handle holds after `call` more than before it."""
    e = QubitVector(N)
    e.initialize_random(3)
    e.norm()  # code objects, the first buffers
    before = device_memory()[0]
    call(e)
    after = device_memory()[0]
    e.close()
    return before - after


def test_marginal_of_many_qubits():
    print("case: memory of a permuted readout", flush=True)
    qubits = list(np.random.default_rng(1).permutation(N))

    def call(e):
        p = e.probabilities(qubits)
        assert abs(p.sum() - 1.0) < 1e-12
    # one double per outcome
    assert taken(call) < 1.5 * ROW


def test_sampling_index_of_every_amplitude():
    print("case: memory of a fine sampling index", flush=True)
    draws = np.random.default_rng(2).random(100)

    def call(e):
        e.set_sample_measure_index_size(N)
        assert e.sample_measure(draws).max() < 1 << N
    # a run and a cumulative sum per amplitude
    assert taken(call) < 2.5 * ROW
