"""Whole-register programs of one workgroup (small fused states, batched
instances, noisy trajectories) around their size classes: below 4 qubits a thread holds
empty slots, 10 is the last single wave, 11 leaves waves without amplitudes, 13
and 14 are the largest."""
from __future__ import annotations

import math

import numpy as np
import pytest

from qclojure_amd import circuit as qc
from qclojure_amd import engine
from qclojure_amd._abi import OP, QSV_FLAG_FUSE

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 3, 4, 5, 9, 10, 11, 12, 13, 14]


def _program(n, rng, count, measure=False):
    rows = []
    names = ["H", "RX", "RY", "RZ", "T", "X"] + (["CNOT", "CZ", "CRX", "CRZ", "SWAP", "ISWAP"] if n > 1 else [])
    names += ["TOFFOLI", "FREDKIN"] if n > 2 else []
    for k in range(count):
        name = names[rng.integers(len(names))]
        q = [int(x) for x in rng.permutation(n)[:3]] + [0, 0, 0]
        used = 3 if name in ("TOFFOLI", "FREDKIN") else 2 if name in ("CNOT", "CZ", "CRX", "CRZ", "SWAP", "ISWAP") else 1
        q = [x if i < used else 0 for i, x in enumerate(q[:3])]
        rows.append((OP[name], q[0], q[1], q[2], 0, float(rng.uniform(0, 2 * math.pi))))
        if measure and k == count // 2:
            rows.append((OP["MEASURE"], 0, 0, 0, 1, 0.0))
    return qc.ops_from_tuples(rows)


@pytest.mark.parametrize("n", [s for s in SIZES if s < 13])
@pytest.mark.parametrize("measure", [False, True])
def test_fused_state(n, measure):
    rng = np.random.default_rng(31 * n + measure)
    first, ops = _program(n, rng, 25), _program(n, rng, 120, measure)
    with engine.DeviceState(n, "c128") as ref, engine.DeviceState(n, "c128") as a, engine.DeviceState(n, "c64") as b:
        for s in (ref, a, b):
            s.apply(first)                       # the fused program starts from a loaded state
        ref.apply(ops, 0, 5)
        a.apply(ops, QSV_FLAG_FUSE, 5)
        b.apply(ops, QSV_FLAG_FUSE, 5)
        exp = ref.download()
        assert np.max(np.abs(a.download() - exp)) < 1e-12
        assert np.max(np.abs(b.download() - exp)) < 1e-5


@pytest.mark.parametrize("n", [1, 4, 11])
@pytest.mark.parametrize("count", [0, 1, 2, 3, 4, 5])
def test_short_fused_programs(n, count):
    """A few gates are launched one by one, on either side of a measurement too."""
    rng = np.random.default_rng(n + 50 * count)
    first, a, b = _program(n, rng, 25), _program(n, rng, count), _program(n, rng, count)
    meas = qc.ops_from_tuples([(OP["MEASURE"], 0, 0, 0, 1, 0.0)])
    for ops in (a, np.concatenate([a, meas, b])):
        with engine.DeviceState(n, "c128") as ref, engine.DeviceState(n, "c128") as s:
            exp = ref.apply(first).apply(ops, 0, 9).download()
            assert np.max(np.abs(s.apply(first).apply(ops, QSV_FLAG_FUSE, 9).download() - exp)) < 1e-13


@pytest.mark.parametrize("precision", ["c128", "c64"])
def test_batched_energies(precision):
    rng = np.random.default_rng(12)
    insts, exp = [], []
    for n in SIZES * 3:
        ops = _program(n, rng, int(rng.integers(0, 90)))
        masks = rng.integers(0, 2 ** n, size=int(rng.integers(1, 140)), dtype=np.uint64)
        coeff = rng.normal(size=len(masks))
        insts.append((n, ops, (masks, coeff)))
        with engine.DeviceState(n, "c128") as s:
            z = s.apply(ops).expect_pauli(["".join("Z" if (int(m) >> q) & 1 else "I" for q in range(n)) for m in masks])
        exp.append(float(np.dot(z, coeff)))
    got = engine.batch_expect_z(insts, precision)
    # FP64 arithmetic for both (13 and 14 qubits of complex128 and complex64 are on either side of
    # the one-workgroup limit, beyond which complex64 states are stored in FP32 between passes)
    scale = np.array([np.sum(np.abs(i[2][1])) for i in insts])
    assert np.max(np.abs(got - exp) / scale) < (1e-12 if precision == "c128" else 1e-6)


def test_batches_of_any_size_in_turn():
    """Programs are staged in memory that the last batch left and gathered anew
    where it is too short; with and without circuits above one workgroup."""
    rng = np.random.default_rng(8)
    for sizes in ([4], [3, 9, 10] * 12, [5], [12] * 30, [2, 15, 7], [11] * 60 + [16], [6, 8]):
        insts, exp = [], []
        for n in sizes:
            ops = _program(n, rng, int(rng.integers(1, 120)))
            masks = rng.integers(0, 2 ** n, size=5, dtype=np.uint64)
            insts.append((n, ops, (masks, np.ones(5))))
            with engine.DeviceState(n, "c128") as s:
                exp.append(sum(s.apply(ops).expect_pauli(["".join("Z" if (int(m) >> q) & 1 else "I" for q in range(n))
                                                          for m in masks])))
        assert np.max(np.abs(engine.batch_expect_z(insts, "c128") - exp)) < 5e-12


# (one workgroup holds 13 qubits of complex128)
@pytest.mark.parametrize("precision,n", [(p, n) for p in ("c128", "c64") for n in SIZES if n < 14 or p == "c64"])
def test_trajectories(oracle, n, precision):
    """Entangling programs with operators that do not keep the norm on every
    qubit, between ones that do; more than 16 sites in all."""
    rng = np.random.default_rng(100 + n)
    ops = _program(n, rng, 40 + n)
    damp, flip, ry = 0.4, 0.3, 0.2
    amp = [np.array([[1, 0], [0, math.sqrt(1 - damp)]]), np.array([[0, math.sqrt(damp)], [0, 0]])]
    bit = [math.sqrt(1 - flip) * np.eye(2), math.sqrt(flip) * np.array([[0, 1], [1, 0]])]
    turn = [np.array([[math.cos(ry), -math.sin(ry)], [math.sin(ry), math.cos(ry)]])]
    sites = [{"after-op": k, "qubit": int(rng.integers(n)) if k >= 2 * n else k % n, "kraus": [amp, bit, turn][k % 3]}
             for k in range(len(ops))]
    T = 6 if n < 11 else 3
    got, states = engine.noisy_trajectories(n, ops, sites, T, 17, precision, n_keep=T)
    exp, fin = oracle.trajectories(n, ops, sites, T, 17, qc.op_u)
    if precision == "c128":
        assert np.array_equal(got, exp)
        assert np.max(np.abs(states - fin)) < 1e-12
    else:   # FP64 arithmetic, amplitudes stored in 32 bits: a shot moves with probability 1e-6
        assert np.array_equal(got, exp)
        assert np.max(np.abs(states - fin)) < 1e-6
