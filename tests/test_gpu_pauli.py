"""Pauli-string expectations against their definition in numpy: register sizes
on both sides of the tiled sweeps' limit, X parts that fit a tile and X parts
that do not, shared X parts, and more strings than one sweep or copy takes."""
from __future__ import annotations

import numpy as np
import pytest

from qclojure_amd import engine

pytestmark = pytest.mark.gpu


def _random_state(n, rng):
    a = rng.normal(size=2 ** n) + 1j * rng.normal(size=2 ** n)
    return a / np.linalg.norm(a)


def _expectation(psi, n, string):
    idx = np.arange(2 ** n, dtype=np.uint64)
    x = s = ny = 0
    for q, ch in enumerate(string):
        b = 1 << (n - 1 - q)
        x |= b if ch in "XY" else 0
        s |= b if ch in "YZ" else 0
        ny += ch == "Y"
    par = idx & np.uint64(s)
    for sh in (32, 16, 8, 4, 2, 1):
        par ^= par >> np.uint64(sh)
    sign = 1.0 - 2.0 * (par & np.uint64(1)).astype(np.float64)
    return ((-1j) ** ny * np.sum(sign * np.conj(psi) * psi[idx ^ np.uint64(x)])).real


def _strings(n, rng):
    out = ["I" * n, "Z" * n, "X" * n, "Y" * n]                       # X parts of full width
    out += ["I" * q + "Z" + "I" * (n - 1 - q) for q in range(n)]
    out += ["I" * q + c + c + "I" * (n - 2 - q) for c in "XYZ" for q in range(n - 1)]
    out += ["".join(rng.choice(list("IXYZ"), n)) for _ in range(12)]
    for _ in range(40):                                               # sparse strings, odd Y counts among them
        t = ["I"] * n
        for q in rng.choice(n, min(n, 3), replace=False):
            t[q] = "XYZ"[rng.integers(3)]
        out.append("".join(t))
    return out


@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n", [1, 2, 7, 11, 12, 18, 19, 20, 21])
def test_expectations(n, precision):
    rng = np.random.default_rng(100 + n)
    psi = _random_state(n, rng)
    if precision == "c64":
        psi = psi.astype(np.complex64).astype(np.complex128)   # what the state holds
    strings = _strings(n, rng)
    with engine.DeviceState(n, precision) as st:
        st.upload(psi)
        got = st.expect_pauli(strings)
    exp = np.array([_expectation(psi, n, s) for s in strings])
    # FP64 sums of at most 2^n terms of total magnitude 1
    assert np.max(np.abs(got - exp)) < 1e-13


@pytest.mark.parametrize("n", [12, 20])
def test_many_strings(n):
    """More Z strings than a sweep, more shared X parts than its units, and more strings than one copy."""
    rng = np.random.default_rng(7)
    psi = _random_state(n, rng)
    strings = ["".join(rng.choice(list("IZ"), n)) for _ in range(300)]
    xs = ["".join(rng.choice(list("IX"), n, p=[0.85, 0.15])) for _ in range(60)]
    for x in xs:   # five strings on each X part
        for _ in range(5):
            strings.append("".join(("XY"[rng.integers(2)] if c == "X" else "IZ"[rng.integers(2)]) for c in x))
    with engine.DeviceState(n, "c128") as st:
        st.upload(psi)
        got = st.expect_pauli(strings)
        again = st.expect_pauli(strings)
    exp = np.array([_expectation(psi, n, s) for s in strings])
    assert np.max(np.abs(got - exp)) < 1e-13
    assert np.array_equal(got, again)   # fixed summation order


@pytest.mark.parametrize("precision", ["c128", "c64"])
@pytest.mark.parametrize("n", [19, 20, 22, 25])
def test_string_by_itself(n, precision):
    """One string in a call, and the one left over after whole chunks of 256."""
    rng = np.random.default_rng(200 + n)
    psi = _random_state(n, rng)
    if precision == "c64":
        psi = psi.astype(np.complex64).astype(np.complex128)
    lone = ["Z" + "I" * (n - 1), "I" * (n - 2) + "XY", "Y" + "I" * (n - 2) + "X", "".join(rng.choice(list("IXYZ"), n))]
    with engine.DeviceState(n, precision) as st:
        st.upload(psi)
        got = [float(st.expect_pauli([s])[0]) for s in lone]
        tail = st.expect_pauli([lone[0]] * 256 + [lone[1]])
    exp = np.array([_expectation(psi, n, s) for s in lone])
    assert np.max(np.abs(np.array(got) - exp)) < 1e-13
    assert np.max(np.abs(tail - np.array([exp[0]] * 256 + [exp[1]]))) < 1e-13
