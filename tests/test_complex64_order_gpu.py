"""complex64 runs keep the order of a gate's products: gate passes sum them in
another one, which moves the state by its rounding and with it the outcomes of
draws and FP64 values."""
import numpy as np
import pytest

from qiskit_aer_amd import AerSimulator, QubitVector
from tests.test_gate_pass_gpu import mixture, wide_mixture

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [12, 13, 17, 20])
@pytest.mark.parametrize("wide", [False, True])
def test_runs_take_no_gate_passes(n, wide):
    print(f"case: complex64 run n={n} wide={wide}", flush=True)
    c = wide_mixture(n, 71, 40) if wide else mixture(n, 72, 150)
    gates = list(c.ops)
    c.measure_all()
    got = AerSimulator(precision="single").run(c, shots=100, seed_simulator=3, save_statevector=True).get_statevector()
    c.ops = gates
    e = QubitVector(n, "single")
    e.set_gate_passes(False)
    e.set_fusion(True, 5, 14)
    e.initialize()
    e.apply_ops(c)
    assert np.array_equal(got, e.copy_to_vector())
    assert e.gate_pass_stats()[0] == 0


def test_handles_take_them_by_default():
    n = 17
    print("case: complex64 handle", flush=True)
    c = wide_mixture(n, 73, 40)
    e = QubitVector(n, "single")
    e.initialize()
    e.apply_ops(c)
    e.synchronize()
    assert e.gate_pass_stats()[0] > 0
    e.set_gate_passes(False)
    before = e.gate_pass_stats()[0]
    e.apply_ops(c)
    e.synchronize()
    assert e.gate_pass_stats()[0] == before


@pytest.mark.parametrize("seed", [1, 2])
def test_gate_passes_are_as_accurate(seed):
    """2x2 gates of U3 in gate passes round no more than in register passes: 20
    layers of brickwork on 23 qubits against the same run in complex128.  The
    norm of the error is that of 2^24 roundings per gate, which another seed
    moves by parts in a thousand."""
    from qiskit_aer_amd import circuits
    n = 23
    print(f"case: complex64 accuracy seed={seed}", flush=True)
    c = circuits.brickwork_u3_cx(n, 20, seed, measure=False)
    d = QubitVector(n)
    d.initialize()
    d.apply_ops(c)
    exact = d.copy_to_vector()
    d.close()
    off = []
    for on in (True, False):
        e = QubitVector(n, "single")
        e.set_gate_passes(on)
        e.initialize()
        e.apply_ops(c)
        off.append(np.linalg.norm(e.copy_to_vector() - exact))
        assert (e.gate_pass_stats()[0] > 0) == on
        e.close()
    assert off[0] < 1.005 * off[1]
