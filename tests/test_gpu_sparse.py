"""States whose tiles are mostly zeros: fused passes leave zero tiles alone, the
gate-by-gate path does not look. Basis states, few active qubits at either end,
uncollapsed and collapsed registers, both arithmetic widths and a batch."""
from __future__ import annotations

import math

import numpy as np
import pytest

from qclojure_amd import circuit as qc
from qclojure_amd import engine
from qclojure_amd._abi import OP, QSV_FLAG_FP64_PASSES, QSV_FLAG_FUSE

pytestmark = pytest.mark.gpu


def _program(qubits, rng, count):
    rows = []
    for _ in range(count):
        a, b = (int(q) for q in rng.choice(qubits, 2, replace=False))
        name = ["H", "RX", "RY", "RZ", "CNOT", "CNOT", "SWAP", "CZ", "X"][rng.integers(9)]
        rows.append((OP[name], a, b if name in ("CNOT", "SWAP", "CZ") else 0, 0, 0, float(rng.uniform(0, 2 * math.pi))))
    return rows


@pytest.mark.parametrize("n", [12, 13, 16, 20, 23])
@pytest.mark.parametrize("where", ["first", "last", "spread", "measured"])
def test_sparse(n, where):
    rng = np.random.default_rng(n)
    some = {"first": range(5), "last": range(n - 5, n), "spread": range(0, n, 3), "measured": range(n)}[where]
    rows = _program(list(some), rng, 60)
    if where == "measured":   # half of the amplitudes go to zero, then more gates
        rows += [(OP["MEASURE"], 0, 0, 0, 0b101, 0.0)] + _program(list(range(n)), rng, 30)
    # FP32 passes end in a norm of one: a register with one tile in use has its sums in one block
    ops = qc.ops_from_tuples(rows)
    with engine.DeviceState(n, "c128") as ref, engine.DeviceState(n, "c128") as a, \
            engine.DeviceState(n, "c64") as f32, engine.DeviceState(n, "c64") as f64:
        ref.apply(ops, 0, 77)
        a.apply(ops, QSV_FLAG_FUSE, 77)
        f32.apply(ops, QSV_FLAG_FUSE, 77)
        f64.apply(ops, QSV_FLAG_FUSE | QSV_FLAG_FP64_PASSES, 77)
        # a hundred gates on amplitudes of at most 1
        assert a.compare(ref)["max_abs_diff"] < 1e-13
        for s in (f32, f64):
            assert s.compare(ref)["max_abs_diff"] < 1e-5
        assert abs(f32.norm2() - 1.0) < 2e-6


@pytest.mark.parametrize("prec,n,arithmetic", [("c128", 24, 64), ("c64", 25, 64), ("c64", 25, 32)])
@pytest.mark.parametrize("start", ["zero", "top", "two", "dense"])
def test_reach(prec, n, arithmetic, start):
    """Large states: the first passes keep track of where amplitudes can be, in
    FP32 passes beside the norms that they hand on (a tile not read has none)."""
    rng = np.random.default_rng(n + len(start))
    rows = []
    if start == "top":
        rows = [(OP["X"], q, 0, 0, 0, 0.0) for q in range(n)]
    elif start == "two":      # two far basis states
        rows = [(OP["H"], 0, 0, 0, 0, 0.0)] + [(OP["CNOT"], 0, q, 0, 0, 0.0) for q in range(1, n)]
    elif start == "dense":
        rows = [(OP["H"], q, 0, 0, 0, 0.0) for q in range(n)]
    first = qc.ops_from_tuples(rows)
    more = [qc.ops_from_tuples(_program(list(qs), rng, 70)) for qs in (range(0, n, 2), range(n))]
    with engine.DeviceState(n, prec) as ref, engine.DeviceState(n, prec) as a:
        for s, flags in ((ref, 0), (a, QSV_FLAG_FUSE | (QSV_FLAG_FP64_PASSES if prec == "c64" and arithmetic == 64 else 0))):
            if len(rows):
                s.apply(first)
            for ops in more:
                s.apply(ops, flags)
        # 140 gates on amplitudes of at most 1; complex64 rounds its stores
        assert a.compare(ref)["max_abs_diff"] < (1e-13 if prec == "c128" else 1e-5)
        # FP32 passes remove their drift, stores that only round leave it
        assert abs(a.norm2() - 1.0) < (1e-12 if prec == "c128" else 2e-6 if arithmetic == 32 else 1e-4)


def test_reach_across_programs():
    """Short programs on one state, as many as use up the passes that may track it
    and more, from a basis state that is set again in between."""
    n = 24
    rng = np.random.default_rng(1)
    with engine.DeviceState(n, "c128") as ref, engine.DeviceState(n, "c128") as a:
        for k in range(8):
            qubits = list(range(n)) if k % 3 else list(range(k, n, 2))
            ops = qc.ops_from_tuples(_program(qubits, rng, 24))
            for s, flags in ((ref, 0), (a, QSV_FLAG_FUSE)):
                if k == 5:
                    s.init_basis(3 * 2 ** 20 + 1)
                s.apply(ops, flags)
            assert a.compare(ref)["max_abs_diff"] < 1e-13
