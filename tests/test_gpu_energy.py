"""Energies of batched states that do not fit one workgroup: the tile transform
at the smallest state of each precision, with strings inside and across tiles
and more strings than a workgroup has threads."""
from __future__ import annotations

import numpy as np
import pytest

from qclojure_amd import circuit as qc
from qclojure_amd import engine
from qclojure_amd._abi import OP

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,sizes", [("c128", (14, 14, 16, 20)), ("c64", (15, 15, 18))])
def test_energy(prec, sizes):
    rng = np.random.default_rng(len(sizes))
    insts, want, room = [], [], []
    for k, n in enumerate(sizes):
        # a product state: <Z-string> is the product of its qubits' cosines
        angles = rng.uniform(0.0, np.pi, n)
        ops = qc.ops_from_tuples([(OP["RY"], q, 0, 0, 0, float(angles[q])) for q in range(n)])
        masks = [rng.choice([False, True], size=n, p=[1 - w, w]) for w in (0.1, 0.5) for _ in range((0, 1, 40, 160)[k])]
        masks += [np.arange(n) == q for q in (0, n - 1)] if k else []
        terms = [(float(rng.normal()), "".join("Z" if b else "I" for b in m)) for m in masks]
        insts.append((n, ops, terms))
        want.append(sum(c * np.prod(np.cos(angles[m])) for (c, _), m in zip(terms, masks)))
        room.append(sum(abs(c) for c, _ in terms))
    got = engine.batch_expect_z(insts, prec)
    # amplitudes carry n roundings of the state's type; the sums are FP64
    eps = 2.0 ** -52 if prec == "c128" else 2.0 ** -23
    for n, g, w, r in zip(sizes, got, want, room):
        assert abs(g - w) <= 4 * n * eps * r, (n, g, w)
