"""What ended handles left for later ones goes back to the device on request,
also while other handles are in use and from several threads."""
import threading

import numpy as np
import pytest

import qiskit_aer_amd as A
from qiskit_aer_amd.qubitvector import device_memory

pytestmark = pytest.mark.gpu


def test_memory_of_ended_handles():
    print("case: release of ended handles", flush=True)
    kept = A.QubitVector(10)
    kept.initialize()
    kept.apply_matrix([3], np.array([[1, 1], [1, -1]]) / np.sqrt(2))
    kept.norm()
    A.release_memory()
    before = device_memory()[0]
    qs = [A.QubitVector(22) for _ in range(4)]  # 64 MiB each
    for q in qs:
        q.initialize()
        q.synchronize()
        q.close()
    held = before - device_memory()[0]
    A.release_memory()
    assert held >= 4 * (64 << 20)
    assert before - device_memory()[0] <= 8 << 20
    A.release_memory()  # nothing left to free
    v = kept.copy_to_vector()
    assert abs(v[0] - v[8]) < 1e-15 and abs(np.linalg.norm(v) - 1) < 1e-14
    kept.close()


def test_release_from_threads():
    print("case: release from threads", flush=True)
    bad = []

    def work(t):
        for k in range(8):
            q = A.QubitVector(3 + (t + k) % 9)
            q.initialize()
            q.apply_mcx([1])
            v = q.copy_to_vector()
            if v[2] != 1 or np.count_nonzero(v) != 1:
                bad.append((t, k))
            q.close()
            if t == 0:
                A.release_memory()

    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
