"""Gates that a fused pass does not run where they stand — CNOTs and swaps that
become index permutations, diagonal gates that wait and are multiplied together —
against the gate-by-gate path, on one tile and on enough tiles to fill the chip."""
from __future__ import annotations

import math

import numpy as np
import pytest

from qclojure_amd import circuit as qc
from qclojure_amd import engine
from qclojure_amd._abi import OP, QSV_FLAG_FP64_PASSES, QSV_FLAG_FUSE

pytestmark = pytest.mark.gpu


def _program(kind, n, rng, count):
    def two():
        return [int(x) for x in rng.choice(n, 2, replace=False)]

    rows = [(OP["RY"], q, 0, 0, 0, float(rng.uniform(0, math.pi))) for q in range(n)]
    for _ in range(count):
        ang = float(rng.uniform(0, 2 * math.pi))
        u = rng.uniform()
        if kind == "permute":        # CNOT chains and swaps with few dense gates between
            a, b = two()
            name = "CNOT" if u < 0.7 else "SWAP" if u < 0.85 else "ISWAP" if u < 0.9 else "H"
            rows.append((OP[name], a, 0 if name == "H" else b, 0, 0, 0.0))
        elif kind == "diagonal":     # phases of every kind, then a dense gate that needs some of them
            a, b = two()
            name = ["RZ", "T", "CZ", "CRZ", "RYDBERG_CPHASE", "PHASE", "RX"][rng.integers(7)]
            rows.append((OP[name], a, b if name[0] == "C" or name[:3] == "RYD" else 0, 0, 0, ang))
        else:                        # both, with controlled dense gates and three-qubit ones
            a, b = two()
            if u < 0.1:
                x, y, z = (int(q) for q in rng.choice(n, 3, replace=False))
                rows.append((OP[["TOFFOLI", "FREDKIN"][rng.integers(2)]], x, y, z, 0, 0.0))
            else:
                name = ["CNOT", "CRX", "CRY", "CRZ", "H", "RY", "RZ", "S", "X", "SWAP", "CY"][rng.integers(11)]
                rows.append((OP[name], a, b if name[0] == "C" or name == "SWAP" else 0, 0, 0, ang))
    return qc.ops_from_tuples(rows)


@pytest.mark.parametrize("kind", ["permute", "diagonal", "mixed"])
@pytest.mark.parametrize("n,count", [(12, 200), (13, 200), (17, 300), (22, 250), (24, 150)])
def test_deferred_gates(kind, n, count):
    rng = np.random.default_rng(n * 7 + len(kind))
    ops = _program(kind, n, rng, count)
    with engine.DeviceState(n, "c128") as ref, engine.DeviceState(n, "c128") as a, \
            engine.DeviceState(n, "c64") as f32, engine.DeviceState(n, "c64") as f64:
        ref.apply(ops)
        a.apply(ops, QSV_FLAG_FUSE)
        f32.apply(ops, QSV_FLAG_FUSE)
        f64.apply(ops, QSV_FLAG_FUSE | QSV_FLAG_FP64_PASSES)
        # FP64: a few hundred roundings of amplitudes of at most 1
        assert a.compare(ref)["max_abs_diff"] < 1e-12
        for s in (f32, f64):
            assert s.compare(ref)["max_abs_diff"] < 1e-5


@pytest.mark.parametrize("n,targets", [(13, 1), (13, 8), (16, 4), (20, 8), (24, 11)])
def test_bits_outside_the_tile(n, targets):
    """Few targets, controls and phases on every qubit: most of them lie outside
    a pass's tile, where a control is a condition and a CNOT shifts the indices."""
    rng = np.random.default_rng(100 * n + targets)
    pool = [int(q) for q in rng.choice(n, targets, replace=False)]
    rows = [(OP["H"], q, 0, 0, 0, 0.0) for q in range(n)]
    for _ in range(250):
        ang = float(rng.uniform(0, 2 * math.pi))
        t = pool[int(rng.integers(targets))]
        c, d = (int(q) for q in rng.choice([q for q in range(n) if q != t], 2, replace=False))
        name = ["CNOT", "CNOT", "CRX", "CRY", "CRZ", "CZ", "RY", "RX", "RZ", "TOFFOLI", "RYDBERG_CPHASE",
                "FREDKIN"][rng.integers(12)]
        if name == "TOFFOLI":
            rows.append((OP[name], c, d, t, 0, 0.0))
        elif name == "FREDKIN":
            rows.append((OP[name], c, t, d, 0, 0.0) if rng.uniform() < 0.2 else (OP["T"], d, 0, 0, 0, 0.0))
        elif name == "RZ":
            rows.append((OP[name], d, 0, 0, 0, ang))
        else:
            rows.append((OP[name], c if name[0] == "C" or name[:3] == "RYD" else t,
                         t if name[0] == "C" or name[:3] == "RYD" else 0, 0, 0, ang))
    ops = qc.ops_from_tuples(rows)
    with engine.DeviceState(n, "c128") as ref, engine.DeviceState(n, "c128") as a, \
            engine.DeviceState(n, "c64") as f32:
        ref.apply(ops)
        a.apply(ops, QSV_FLAG_FUSE)
        f32.apply(ops, QSV_FLAG_FUSE)
        # as above: a few hundred roundings of amplitudes of at most 1
        assert a.compare(ref)["max_abs_diff"] < 1e-12
        assert f32.compare(ref)["max_abs_diff"] < 1e-5


def test_diagonal_entries_change_the_plan():
    """Two batches of one structure: the diagonal gates of the first are phases,
    which need no tile bit, those of the second are not."""
    n = 16
    rng = np.random.default_rng(3)
    angles = rng.uniform(0, math.pi, n)
    terms = [(1.0, "".join("Z" if q == k else "I" for q in range(n))) for k in range(n)]
    for d0 in (1j, 0.5):
        ops = np.concatenate([qc.ops_from_tuples([(OP["RY"], q, 0, 0, 0, float(angles[q])) for q in range(n)])] +
                             [qc.op_u(q, np.diag([d0, 1.0])) for q in range(n)] +
                             [qc.ops_from_tuples([(OP["RX"], q, 0, 0, 0, 0.3) for q in range(n)])])
        with engine.DeviceState(n, "c128") as ref:
            ref.apply(ops)
            want = sum(ref.expect_pauli([s for _, s in terms]))
        got = engine.batch_expect_z([(n, ops, terms)] * 2, "c128")
        # a sum of 16 values of at most 1 after 48 gates
        assert np.max(np.abs(np.asarray(got) - want)) < 1e-12


@pytest.mark.parametrize("n", [5, 12, 16])
@pytest.mark.parametrize("entry", range(4))
def test_nan_entry_is_not_dropped(n, entry):
    """A general 2x2 with one NaN entry leaves NaN where the gate-by-gate path does."""
    u = np.array([[0.6, 0.8j], [0.8j * np.exp(0.3j), 0.6 * np.exp(0.3j)]])
    u[entry // 2, entry % 2] = complex(math.nan, 0.1)
    first = qc.ops_from_tuples([(OP["RY"], q, 0, 0, 0, 0.5 + q) for q in range(n)])
    # more than a program of a gate or two, none of them folded into the general one
    ops = np.concatenate([qc.op_u(1, u), qc.ops_from_tuples([(OP["RY"], q, 0, 0, 0, 0.3) for q in range(2, n)])])
    with engine.DeviceState(n, "c128") as ref, engine.DeviceState(n, "c128") as a:
        want = np.isnan(ref.apply(first).apply(ops).download())
        assert np.any(want)
        assert np.array_equal(np.isnan(a.apply(first).apply(ops, QSV_FLAG_FUSE).download()), want)


@pytest.mark.parametrize("n,layers", [(5, 100), (10, 60), (13, 20)])
def test_general_unitaries_are_the_callers(n, layers):
    """Layers of general one-qubit unitaries: fused passes are as near to the
    exact result as one gate after the other."""
    rng = np.random.default_rng(n)
    psi = np.zeros(2 ** n, dtype=np.clongdouble)
    psi[0] = 1
    i = np.arange(2 ** n)
    ops = []
    for _ in range(layers):
        for q in range(n):
            a, b, c = rng.uniform(0, 2 * math.pi, 3)
            u = np.array([[math.cos(a / 2), -np.exp(1j * c) * math.sin(a / 2)],
                          [np.exp(1j * b) * math.sin(a / 2), np.exp(1j * (b + c)) * math.cos(a / 2)]])
            ops.append(qc.op_u(q, u))
            v, w = psi.reshape(2 ** q, 2, -1), u.astype(np.clongdouble)
            v[:, 0], v[:, 1] = w[0, 0] * v[:, 0] + w[0, 1] * v[:, 1], w[1, 0] * v[:, 0] + w[1, 1] * v[:, 1]
        perm = [int(q) for q in rng.permutation(n)]
        for x, y in zip(perm[::2], perm[1::2]):
            ops.append(qc.ops_from_tuples([(OP["CZ"], x, y, 0, 0, 0.0)]))
            psi[((i >> (n - 1 - x)) & (i >> (n - 1 - y)) & 1) == 1] *= -1
    ops = np.concatenate(ops)
    err = []
    for flags in (0, QSV_FLAG_FUSE):
        with engine.DeviceState(n, "c128") as s:
            err.append(float(np.linalg.norm(s.apply(ops, flags).download() - psi)))
    # the same roundings in another order: two such sums over hundreds of gates agree within a quarter
    assert err[1] < 1.25 * err[0], err
