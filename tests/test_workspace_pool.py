"""The pool of ended handles' buffers, compiled for the host on a fake HIP
runtime (tests/adaptor/fake_hip): its bounds, what a failed allocation does,
and several devices.  No device needed."""
import pathlib
import shutil
import subprocess

import pytest

HERE = pathlib.Path(__file__).resolve().parent
CSRC = HERE.parent / "qiskit_aer_amd" / "csrc"


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    out = tmp_path_factory.mktemp("pool") / "workspace_pool"
    r = subprocess.run(["g++", "-std=c++17", "-Wall", "-pthread", f"-I{HERE / 'adaptor' / 'fake_hip'}", f"-I{CSRC}",
                        str(HERE / "adaptor" / "workspace_pool.cpp"), "-o", str(out)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return out


@pytest.mark.parametrize("case", ["bounded", "out_of_memory", "devices", "leases"])
def test_pool(program, case):
    r = subprocess.run([str(program), case], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
