"""Shots against the inverse CDF in extended precision, on register sizes around
the sampler's chunk (2^10 amplitudes) and group (2^20 amplitudes) limits."""
from __future__ import annotations

import threading

import numpy as np
import pytest

from qclojure_amd import engine

pytestmark = pytest.mark.gpu


def _expected(psi, shots, seed):
    cum = np.cumsum((psi.real.astype(np.longdouble) ** 2 + psi.imag.astype(np.longdouble) ** 2))
    u = np.array([engine.uniform(seed, k) for k in range(shots)], dtype=np.longdouble)
    return np.minimum(np.searchsorted(cum, u * cum[-1], side="left"), len(psi) - 1).astype(np.uint64)


@pytest.mark.parametrize("n,shots", [(1, 9), (3, 100), (6, 300), (9, 500), (10, 1000), (11, 1000), (16, 2000),
                                     (20, 2000), (21, 2000), (22, 70000),
                                     # enough shots for the kernel that reads less and waits more
                                     (1, 2049), (4, 3000), (7, 5000), (10, 2049), (11, 4000), (15, 9000), (20, 2048),
                                     (20, 2049), (21, 6000)])
@pytest.mark.parametrize("precision", ["c128", "c64"])
def test_shots(n, shots, precision):
    rng = np.random.default_rng(n)
    psi = rng.normal(size=2 ** n) + 1j * rng.normal(size=2 ** n)
    psi *= rng.uniform(size=2 ** n) < 0.7    # zeros between
    psi[rng.integers(2 ** n)] += 1.0         # never all zero
    psi /= np.linalg.norm(psi)
    if precision == "c64":
        psi = psi.astype(np.complex64).astype(np.complex128)
    with engine.DeviceState(n, precision) as st:
        st.upload(psi)
        got = st.sample(shots, 11)
        few = st.sample(5, 11)
    # a rounding of the FP64 prefix moves a shot with probability 2^n * 1e-15
    assert np.array_equal(got, _expected(psi, shots, 11))
    assert np.array_equal(few, got[:5])


@pytest.mark.parametrize("index", [0, 1023, 1024, 2 ** 20 - 1, 2 ** 20, 2 ** 21 - 1])
def test_basis_states(index):
    with engine.DeviceState(21, "c128") as st:
        assert set(st.init_basis(index).sample(64, 3).tolist()) == {index}


def test_readers_in_threads():
    """Several threads read one state: shots of different counts (the kept buffer
    grows under way), expectations and norms, each as from one thread alone."""
    n = 18
    rng = np.random.default_rng(n)
    psi = rng.normal(size=2 ** n) + 1j * rng.normal(size=2 ** n)
    psi /= np.linalg.norm(psi)
    strings = ["I" * q + p + "I" * (n - 1 - q) for q in range(n) for p in "XYZ"]
    with engine.DeviceState(n, "c128") as st, engine.DeviceState(n, "c128") as alone:
        st.upload(psi)
        alone.upload(psi)
        jobs = [(lambda s, k=k: s.sample(700 + 500 * k, k)) for k in range(4)]
        jobs += [lambda s: s.expect_pauli(strings), lambda s: s.expect_pauli(strings[::-1]),
                 lambda s: np.array([s.norm2(), s.expect_1q(3, [[1, 2j], [-2j, 3]]).real, s.inner(alone).real])]
        wrong = []

        def work(job, want):
            for _ in range(40):
                if not np.array_equal(job(st), want):
                    wrong.append(job)

        threads = [threading.Thread(target=work, args=(j, j(alone))) for j in jobs]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not wrong
