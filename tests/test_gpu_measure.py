"""Outcome weights and collapse: which of the measured bits lie in a lane, in a
wave, among the bits a thread walks (its outcomes in runs of one amplitude and more,
up to eight in a row) or above them; states smaller than a block."""
from __future__ import annotations

import numpy as np
import pytest

from qclojure_amd import engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["c128", "c64"])
@pytest.mark.parametrize("n,qubits", [
    (1, [0]), (2, [0, 1]), (7, [6]), (8, [0, 7]), (9, [0]), (12, list(range(12))), (14, [0, 1]), (14, [12, 13]),
    (15, [0, 5, 6, 9, 14]), (17, [1, 2, 3, 4, 5, 6, 7, 8]), (18, list(range(6, 18))), (18, list(range(0, 14))),
    (12, [3]), (13, list(range(8))), (16, [4, 6]), (17, [5, 7, 16]), (20, list(range(12))), (21, [9, 12]),
    (25, [0, 12, 24]), (10, [0, 1]), (10, [1]), (11, [0, 2]), (19, list(range(11)) + [17]), (21, list(range(12))),
    (22, list(range(12))), (22, [3, 9, 13]), (22, list(range(6, 15))), (23, [2, 3, 15, 22]),
])
def test_measure(prec, n, qubits):
    rng = np.random.default_rng(n * 31 + len(qubits))
    dt, eps = (np.complex128, 2.0 ** -52) if prec == "c128" else (np.complex64, 2.0 ** -23)
    psi = (rng.standard_normal(1 << n) + 1j * rng.standard_normal(1 << n))
    psi = (psi / np.linalg.norm(psi)).astype(dt)
    m = len(qubits)
    idx = np.arange(1 << n, dtype=np.int64)
    outcome = np.zeros(1 << n, dtype=np.int64)
    for j, q in enumerate(sorted(qubits)):
        outcome |= ((idx >> (n - 1 - q)) & 1) << j
    w = np.bincount(outcome, weights=np.abs(psi.astype(np.complex128)) ** 2, minlength=1 << m)
    with engine.DeviceState(n, prec) as s:
        s.upload(psi)
        o, p = s.measure_qubits(qubits, 0.37)
        got = s.download()
    # FP64 sums of 2^n positive numbers that add up to 1, in any order
    assert np.max(np.abs(p - w)) < 1e-13
    assert o == min(int(np.searchsorted(np.cumsum(p), 0.37 * p.sum())), (1 << m) - 1)
    keep = outcome == o
    assert not got[~keep].any()
    assert np.max(np.abs(got[keep] - psi[keep] / np.sqrt(p[o]))) <= 4 * eps * np.max(np.abs(psi)) / np.sqrt(p[o])
