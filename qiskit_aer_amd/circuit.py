"""A minimal circuit container with Aer's operation names.

``Circuit`` records operations the way Aer's ``AerCircuit`` holds them after
``aer_compiler.assemble_circuits`` (gate name, qubits, real parameters;
``unitary`` / ``diagonal`` matrices; ``measure`` with memory bits), and packs
them into the ``aerhip_op`` wire format of include/aerhip.h.
"""
from __future__ import annotations

import array
import ctypes as C
import itertools
from dataclasses import dataclass, field
from typing import Optional, Sequence

import numpy as np

from . import _lib as L


@dataclass
class Op:
    type: int
    name: str = ""
    qubits: tuple = ()
    params: tuple = ()
    matrix: Optional[np.ndarray] = None  # complex, column-major vectorised or diagonal
    label: Optional[str] = None          # Pauli label
    memory: tuple = ()


@dataclass
class Circuit:
    num_qubits: int
    num_clbits: int = 0
    global_phase: float = 0.0
    ops: list = field(default_factory=list)

    # generic ------------------------------------------------------------------
    def gate(self, name: str, qubits: Sequence[int], params: Sequence[float] = ()) -> "Circuit":
        for q in qubits:
            if not 0 <= int(q) < self.num_qubits:
                raise ValueError(f"qubit {q} out of range")
        self.ops.append(Op(L.OP_GATE, name, tuple(int(q) for q in qubits),
                           tuple(float(p) for p in params)))
        return self

    def unitary(self, matrix, qubits: Sequence[int]) -> "Circuit":
        m = np.asarray(matrix, dtype=np.complex128)
        d = 1 << len(qubits)
        if m.shape != (d, d):
            raise ValueError("unitary has the wrong shape")
        self.ops.append(Op(L.OP_MATRIX, "unitary", tuple(int(q) for q in qubits),
                           matrix=np.ascontiguousarray(m.reshape(-1, order="F"))))
        return self

    def diagonal(self, diag, qubits: Sequence[int]) -> "Circuit":
        d = np.ascontiguousarray(np.asarray(diag, dtype=np.complex128).reshape(-1))
        if d.size != 1 << len(qubits):
            raise ValueError("diagonal has the wrong size")
        self.ops.append(Op(L.OP_DIAGONAL, "diagonal", tuple(int(q) for q in qubits), matrix=d))
        return self

    def initialize(self, state, qubits: Sequence[int]) -> "Circuit":
        s = np.ascontiguousarray(np.asarray(state, dtype=np.complex128).reshape(-1))
        self.ops.append(Op(L.OP_INITIALIZE, "initialize", tuple(int(q) for q in qubits), matrix=s))
        return self

    def measure(self, qubits: Sequence[int], clbits: Sequence[int]) -> "Circuit":
        qubits, clbits = list(qubits), list(clbits)
        self.num_clbits = max(self.num_clbits, max(clbits) + 1)
        self.ops.append(Op(L.OP_MEASURE, "measure", tuple(qubits), memory=tuple(clbits)))
        return self

    def measure_all(self) -> "Circuit":
        self.num_clbits = max(self.num_clbits, self.num_qubits)
        for q in range(self.num_qubits):
            self.ops.append(Op(L.OP_MEASURE, "measure", (q,), memory=(q,)))
        return self

    def reset(self, qubits) -> "Circuit":
        self.ops.append(Op(L.OP_RESET, "reset", tuple(np.atleast_1d(qubits).tolist())))
        return self

    def barrier(self, *qubits) -> "Circuit":
        q = qubits or tuple(range(self.num_qubits))
        self.ops.append(Op(L.OP_BARRIER, "barrier", tuple(q)))
        return self

    def save_statevector(self) -> "Circuit":
        self.ops.append(Op(L.OP_SAVE_STATEVECTOR, "save_statevector", tuple(range(self.num_qubits))))
        return self

    def pauli(self, label: str, qubits: Sequence[int]) -> "Circuit":
        self.ops.append(Op(L.OP_GATE, "pauli", tuple(qubits), label=label))
        return self

    # named gates (Aer spellings) ----------------------------------------------
    def __getattr__(self, name):
        if name.startswith("_"):
            raise AttributeError(name)
        nparams = {"u3": 3, "u": 3, "u2": 2, "u1": 1, "p": 1, "rx": 1, "ry": 1, "rz": 1,
                   "r": 2, "cp": 1, "crx": 1, "cry": 1, "crz": 1, "cu1": 1, "cu2": 2,
                   "cu3": 3, "cu": 4, "rxx": 1, "ryy": 1, "rzz": 1, "rzx": 1, "mcp": 1,
                   "mcphase": 1, "mcu1": 1, "mcu2": 2, "mcu3": 3, "mcu": 4, "mcr": 2,
                   "mcrx": 1, "mcry": 1, "mcrz": 1}.get(name, 0)

        def method(*args):
            params, qubits = args[:nparams], args[nparams:]
            if len(qubits) == 1 and isinstance(qubits[0], (list, tuple)):
                qubits = qubits[0]
            return self.gate(name, qubits, params)
        return method

    def count_gates(self) -> int:
        return sum(1 for o in self.ops if o.type in (L.OP_GATE, L.OP_MATRIX, L.OP_DIAGONAL))

    # wire format ---------------------------------------------------------------
    def pack(self):
        """Returns (ctypes array of AerhipOp, keepalive list).

        The qubits, real parameters and names of all ops go into three flat
        buffers and the records are filled column by column, so packing costs
        a few Python-level passes over the op list rather than a handful of
        small arrays per op."""
        ops = self.ops
        nops = len(ops)
        arr = (L.AerhipOp * nops)()
        keep = []
        if nops == 0:
            return arr, keep
        # One list per attribute, into arrays of machine words (several times
        # faster than numpy reading the objects), and numpy for the rest.
        rec = np.frombuffer(arr, dtype=_OP_DTYPE)
        chain = itertools.chain.from_iterable
        types = [o.type for o in ops]
        rec["type"] = _words("i", types)
        only_gates = types.count(L.OP_GATE) == nops
        # qubits
        qubits = [o.qubits for o in ops]
        nq = _words("q", list(map(len, qubits)))
        qflat, at = _buffer("Q", list(chain(qubits)) + [0])
        keep.append(qflat)
        rec["num_qubits"] = nq
        rec["qubits"] = at + 8 * (np.cumsum(nq) - nq)
        # real parameters: gate angles, then complex matrices as (re, im) pairs
        params = [o.params for o in ops]
        mats = []
        if not only_gates:
            params = [p if t == L.OP_GATE else () for p, t in zip(params, types)]
            mats = [i for i, t in enumerate(types) if t != L.OP_GATE and ops[i].matrix is not None]
        npar = _words("q", list(map(len, params)))
        pflat, at = _buffer("d", list(chain(params)) + [0.0])
        keep.append(pflat)
        rec["num_params"] = npar
        rec["params"] = at + 8 * (np.cumsum(npar) - npar)
        for i in mats:
            m = ops[i].matrix
            if m.ndim > 1 and m.size != m.shape[-1]:
                raise ValueError("the matrix of an op is a vector, its columns one after the other")
            m = np.array(m, dtype=np.complex128)  # packed ops do not follow later changes
            keep.append(m)
            rec["num_params"][i] = m.size
            rec["params"][i] = m.ctypes.data
        # names: one NUL-terminated copy of each distinct name
        names = [o.name for o in ops]
        distinct = sorted(set(names))
        blob = b"".join(nm.encode() + b"\0" for nm in distinct)
        nbuf = array.array("B", blob + b"\0")
        keep.append(nbuf)
        addr, at = {}, nbuf.buffer_info()[0]
        for nm in distinct:
            addr[nm] = at
            at += len(nm.encode()) + 1
        rec["name"] = _words("Q", list(map(addr.__getitem__, names)))
        # Pauli labels and measure clbits (rare)
        for i in [i for i, o in enumerate(ops) if o.label is not None or o.memory]:
            op = ops[i]
            if op.label is not None:
                lab = op.label.encode()
                keep.append(lab)
                arr[i].string_param = lab
            if op.memory:
                m = np.ascontiguousarray(np.asarray(op.memory, dtype=np.uint64))
                keep.append(m)
                arr[i].memory = m.ctypes.data_as(C.POINTER(C.c_uint64))
        return arr, keep


def _words(code: str, values: list) -> np.ndarray:
    return np.frombuffer(array.array(code, values), dtype=code)


def _buffer(code: str, values: list):
    """The values as machine words, and their address.  array.array reads a list
    several times faster than numpy, but refuses qubits given as floats (2.0),
    bools or text, which numpy converts."""
    try:
        words = array.array(code, values)
        return words, words.buffer_info()[0]
    except TypeError:
        words = np.fromiter(values, dtype=code, count=len(values))
        return words, words.ctypes.data


# Field layout of AerhipOp (include/aerhip.h) for filling packed records.
_OP_DTYPE = np.dtype({
    "names": ["type", "num_qubits", "name", "qubits", "num_params", "reserved", "params",
              "string_param", "memory"],
    "formats": ["<i4", "<u4", "<u8", "<u8", "<u4", "<u4", "<u8", "<u8", "<u8"],
    "offsets": [L.AerhipOp.type.offset, L.AerhipOp.num_qubits.offset, L.AerhipOp.name.offset,
                L.AerhipOp.qubits.offset, L.AerhipOp.num_params.offset, L.AerhipOp.reserved.offset,
                L.AerhipOp.params.offset, L.AerhipOp.string_param.offset, L.AerhipOp.memory.offset],
    "itemsize": C.sizeof(L.AerhipOp),
})
