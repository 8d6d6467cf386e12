"""The work a user of this framework has it do, as a list of measurable cases.

listed() gives the named cases, draw() one more of the same ranges; prepare()
makes what a program holds before the call (device states, packed batches, a
running server), run() is one pass through the public entry points and returns
what that program reads, work() the bytes and operations a pass cannot do
without, and exact() the same outputs from plain torch / numpy in 64 bits.

Kinds of cases:
  layers   a circuit of random layers (H, RX, RY or RZ on every qubit, CNOTs on
           a random matching) from |0..0>, then its results: the state vector
           of a small register, otherwise shots and every qubit's <Z>
  qaoa     one MaxCut ansatz on a graph of any size and the <ZZ> of its edges
  results  result extraction from a state in HBM: shots, the terms of a
           Heisenberg chain, one-qubit observables
  measure  a copy of a state, a mid-circuit measurement of some of its qubits
           and shots of the collapsed state
  batch    many QAOA instances in one call, the form of an optimiser's
           parallel evaluations
  noisy    noisy trajectories of the hardware simulator
  serve    requests of mixed sizes through the serving loop
  expm     exp(-iHt) of a dense Hermitian matrix by the linear-algebra backend

complex64 states are asked for amplitudes and expectation values, returned in
32 bits, the precision the path carries; shots are taken of complex128 states,
where rounding does not move a shot from one outcome to its neighbour.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from qclojure_amd import algorithms, engine, hardware, la, workloads
from qclojure_amd import _abi
from qclojure_amd import circuit as circuits

AMPLITUDES_UP_TO = 14   # registers small enough that a program reads the whole state vector


def listed() -> list[dict]:
    return [
        # a teaching-size circuit: all latency and launches
        {"name": "layers_5q", "kind": "layers", "n": 5, "layers": 4, "precision": "c128", "fuse": True, "shots": 100},
        # the 12-qubit, 20-layer circuit the benchmark projects for the reference's own algorithm
        {"name": "layers_12q", "kind": "layers", "n": 12, "layers": 20, "precision": "c128", "fuse": True,
         "shots": 1024},
        # an ordinary simulator job of an odd size, the state in the last-level cache
        {"name": "layers_19q", "kind": "layers", "n": 19, "layers": 10, "precision": "c128", "fuse": True,
         "shots": 1000},
        # a large job: 2 GiB of state in HBM, fused passes
        {"name": "layers_27q", "kind": "layers", "n": 27, "layers": 6, "precision": "c128", "fuse": True,
         "shots": 1000},
        # the same circuits gate by gate (the default flags)
        {"name": "gates_25q", "kind": "layers", "n": 25, "layers": 1, "precision": "c128", "fuse": False,
         "shots": 1000},
        # one large variational evaluation in complex64 (FP32 passes)
        {"name": "qaoa_26q_c64", "kind": "qaoa", "n": 26, "p": 2, "precision": "c64", "fuse": True},
        # everything a result map asks of a final state
        {"name": "results_25q", "kind": "results", "n": 25, "precision": "c128", "shots": 4096},
        # mid-circuit measurement of three qubits
        {"name": "measure_24q", "kind": "measure", "n": 24, "m": 3, "precision": "c128", "shots": 256},
        # an optimiser's population: 512 instances of 8 to 20 qubits, complex64 states
        {"name": "batch_512_c64", "kind": "batch", "count": 512, "n_min": 8, "n_max": 20, "precision": "c64"},
        # the hardware simulator's shots: one trajectory each
        {"name": "noisy_11q", "kind": "noisy", "n": 11, "layers": 3, "trajectories": 1000, "precision": "c128"},
        # a burst of requests, 10 to 22 qubits, depth 10 to 40
        {"name": "serve_24", "kind": "serve", "requests": 24, "n_min": 10, "n_max": 22, "shots": 1000},
        # the evolution operator of a six-qubit Hamiltonian
        {"name": "expm_64", "kind": "expm", "n": 64},
    ]


def draw(rng) -> dict:
    kind = rng.choice(["layers", "layers", "layers", "qaoa", "results", "measure", "batch", "noisy", "serve", "expm"])
    if kind == "layers":
        fuse = rng.random() < 0.7
        precision = "c64" if rng.random() < 0.25 else "c128"
        # complex64 registers whose amplitudes are read; others over the whole range
        n = rng.randint(2, AMPLITUDES_UP_TO) if precision == "c64" else rng.randint(2, 27 if fuse else 25)
        most = (6 if fuse else 1) * 2.0 ** ((27 if fuse else 25) - n)
        layers = int(round(math.exp(rng.uniform(0.0, math.log(max(1.0, min(30.0, most)))))))
        return {"kind": "layers", "n": n, "layers": layers, "precision": precision, "fuse": fuse,
                "shots": 0 if precision == "c64" else rng.randint(1, 2000)}
    if kind == "qaoa":
        n = rng.randint(4, 26)
        return {"kind": "qaoa", "n": n, "p": rng.randint(1, 2 if n > 24 else 4),
                "precision": rng.choice(["c64", "c128"]) if n < 26 else "c64", "fuse": True}
    if kind == "results":
        return {"kind": "results", "n": rng.randint(6, 25), "precision": "c128",
                "shots": int(math.exp(rng.uniform(math.log(100), math.log(20000))))}
    if kind == "measure":
        n = rng.randint(4, 24)
        return {"kind": "measure", "n": n, "m": rng.randint(1, min(n, 8)), "precision": "c128",
                "shots": rng.randint(1, 1000)}
    if kind == "batch":
        lo = rng.randint(4, 12)
        return {"kind": "batch", "count": int(math.exp(rng.uniform(math.log(8), math.log(512)))), "n_min": lo,
                "n_max": rng.randint(lo, 20), "precision": rng.choice(["c64", "c64", "c128"])}
    if kind == "noisy":
        n = rng.randint(2, 13)
        return {"kind": "noisy", "n": n, "layers": rng.randint(1, 4),
                "trajectories": max(8, min(2000, int(1000 * 2.0 ** (11 - n)))) // rng.randint(1, 4),
                "precision": "c128"}
    if kind == "serve":
        lo = rng.randint(5, 14)
        return {"kind": "serve", "requests": rng.randint(4, 24), "n_min": lo, "n_max": rng.randint(lo + 1, 22),
                "shots": rng.randint(100, 1000)}
    return {"kind": "expm", "n": rng.randint(2, 64)}


# ---- inputs -------------------------------------------------------------------
def _graph(n: int, rng) -> list:
    """A ring of n vertices with n // 2 random chords, unit weights."""
    edges = {(i, (i + 1) % n) if i + 1 < n else (0, n - 1) for i in range(n)}
    want = min(n + n // 2, n * (n - 1) // 2)
    while len(edges) < want:
        a, b = sorted(int(x) for x in rng.choice(n, 2, replace=False))
        edges.add((a, b))
    return [[a, b, 1.0] for a, b in sorted(edges)]


def _qaoa(n: int, p: int, rng) -> dict:
    graph = _graph(n, rng)
    return {"n": n, "graph": graph, "hamiltonian": algorithms.max_cut_hamiltonian(graph, n),
            "params": [float(x) for x in rng.uniform(0.0, math.pi, 2 * p)]}


def _batch_instances(case: dict, seed: int) -> list[dict]:
    rng = np.random.default_rng(seed)
    return [_qaoa(int(rng.integers(case["n_min"], case["n_max"] + 1)), int(rng.integers(1, 5)), rng)
            for _ in range(case["count"])]


def _zz_strings(inst: dict) -> list[str]:
    return [t["pauli-string"] for t in inst["hamiltonian"] if "Z" in t["pauli-string"]]


def _z_strings(n: int) -> list[str]:
    return ["I" * q + "Z" + "I" * (n - 1 - q) for q in range(n)]


def _chain_strings(n: int) -> list[str]:
    """XX, YY and ZZ on neighbours and Z on every site: a Heisenberg chain in a field."""
    return ["I" * q + c + c + "I" * (n - 2 - q) for c in "XYZ" for q in range(n - 1)] + _z_strings(n)


def _observables(n: int, rng) -> list:
    """Hermitian one-qubit observables and their qubits."""
    out = []
    for _ in range(3):
        a = rng.normal(size=(2, 2)) + 1j * rng.normal(size=(2, 2))
        out.append((int(rng.integers(n)), a + a.conj().T))
    return out


def _hermitian(n: int, seed: int) -> np.ndarray:
    rng = np.random.default_rng(seed)
    a = rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))
    return (a + a.conj().T) / math.sqrt(8.0 * n)


_NOISE = {"gate-noise": {"h": {"noise-type": "depolarizing", "noise-strength": 0.02},
                         "rx": {"noise-type": "depolarizing", "noise-strength": 0.02},
                         "ry": {"noise-type": "amplitude-damping", "noise-strength": 0.02},
                         "rz": {"noise-type": "phase-damping", "noise-strength": 0.02},
                         "cnot": {"noise-type": "depolarizing", "noise-strength": 0.05}}}


def prepare(case: dict, seed: int) -> dict:
    kind, st = case["kind"], {"case": case, "seed": int(seed)}
    rng = np.random.default_rng(seed)
    if kind == "layers":
        st["state"] = engine.DeviceState(case["n"], case["precision"])
        st["ops"] = workloads.random_layer_ops(case["n"], case["layers"], seed)
        st["flags"] = _abi.QSV_FLAG_FUSE if case["fuse"] else 0
        st["strings"] = _z_strings(case["n"])
    elif kind == "qaoa":
        inst = _qaoa(case["n"], case["p"], rng)
        st["state"] = engine.DeviceState(case["n"], case["precision"])
        st["ops"] = workloads.qaoa_ops(inst)
        st["flags"] = _abi.QSV_FLAG_FUSE if case["fuse"] else 0
        st["strings"] = _zz_strings(inst)
    elif kind in ("results", "measure"):
        st["state"] = engine.DeviceState(case["n"], case["precision"])
        st["state"].apply(workloads.random_layer_ops(case["n"], 2, seed), _abi.QSV_FLAG_FUSE)
        st["state"].sync()
        if kind == "results":
            st["strings"] = _chain_strings(case["n"])
            st["observables"] = _observables(case["n"], rng)
        else:
            st["work"] = engine.DeviceState(case["n"], case["precision"])
            st["qubits"] = sorted(int(q) for q in rng.choice(case["n"], case["m"], replace=False))
            st["u"] = float(rng.uniform())
    elif kind == "batch":
        insts = [(i["n"], workloads.qaoa_ops(i), workloads.qaoa_terms(i)) for i in _batch_instances(case, seed)]
        st["batch"] = engine.PackedBatch(insts, case["precision"])
        engine.init()
    elif kind == "noisy":
        c = workloads.random_layer_circuit(case["n"], case["layers"], seed)
        st["ops"], st["sites"] = hardware.program_with_noise(c, _NOISE)
        engine.init()
    elif kind == "serve":
        reqs = workloads.serving_stream(case["requests"], 1000.0, seed, case["n_min"], case["n_max"], 10, 40,
                                        case["shots"])
        st["requests"] = [(r["n"], workloads.random_layer_ops(r["n"], max(1, r["depth"] // 2), r["seed"]), r["seed"])
                          for r in reqs]
        st["server"] = engine.Server(precision="c128")
    else:
        st["backend"] = la.create_backend("hip")
        st["a"] = st["backend"].matrix_to_backend(-1j * _hermitian(case["n"], seed))
    return st


def run(st: dict):
    case = st["case"]
    kind = case["kind"]
    if kind == "layers":
        s = st["state"].init_basis(0).apply(st["ops"], st["flags"], st["seed"])
        out = {}
        if case["n"] <= AMPLITUDES_UP_TO:
            amps = s.download()
            out["amplitudes"] = amps.astype(np.complex64) if case["precision"] == "c64" else amps
        else:
            out["z"] = s.expect_pauli(st["strings"])
        if case["shots"]:
            out["shots"] = s.sample(case["shots"], st["seed"])
        return out
    if kind == "qaoa":
        zz = st["state"].init_basis(0).apply(st["ops"], st["flags"], st["seed"]).expect_pauli(st["strings"])
        return {"zz": zz.astype(np.float32) if case["precision"] == "c64" else zz}
    if kind == "results":
        s = st["state"]
        return {"shots": s.sample(case["shots"], st["seed"]), "terms": s.expect_pauli(st["strings"]),
                "observables": np.array([s.expect_1q(q, m) for q, m in st["observables"]])}
    if kind == "measure":
        w = st["work"].copy_from(st["state"])
        outcome, probs = w.measure_qubits(st["qubits"], st["u"])
        return {"outcome": outcome, "probabilities": probs, "shots": w.sample(case["shots"], st["seed"])}
    if kind == "batch":
        e = st["batch"].run()
        return {"energies": e.astype(np.float32) if case["precision"] == "c64" else e}
    if kind == "noisy":
        outcomes, _ = engine.noisy_trajectories(case["n"], st["ops"], st["sites"], case["trajectories"], st["seed"],
                                                case["precision"])
        return {"outcomes": outcomes}
    if kind == "serve":
        srv = st["server"]
        ids = [srv.submit(n, ops, case["shots"], seed) for n, ops, seed in st["requests"]]
        return {"shots": np.concatenate([srv.wait(i, case["shots"])[1] for i in ids])}
    return {"exp": st["backend"].matrix_exp(st["a"]).to_numpy()}


# ---- what a pass cannot do without ------------------------------------------------
def _layer_flops(n: int, layers: int) -> float:
    """Real operations of random layers on 2^n amplitudes: RX, RY and H take 6 an
    amplitude (two real multiply-adds a component pair), RZ a complex product
    (6), CNOT none."""
    return 6.0 * n * layers * 2.0 ** n


def _qaoa_flops(n: int, p: int) -> float:
    """Per layer a phase for each of the 3n/2 edges and an RX on every qubit, 6 each."""
    return 6.0 * (n + n // 2 + n) * p * 2.0 ** n


def work(case: dict) -> dict:
    kind = case["kind"]
    item = 8.0 if case.get("precision") == "c64" else 16.0
    if kind == "layers":
        n = case["n"]
        size = item * 2.0 ** n
        if case["fuse"]:
            nbytes = 2.0 * size   # the state written by the circuit and read by its results
        else:
            # gate by gate: every amplitude a gate changes is read and written (CNOTs half)
            nbytes = 2.0 * size * case["layers"] * (n + 0.5 * (n // 2)) + size
        return {"bytes": nbytes + 8.0 * case["shots"], "flops": _layer_flops(n, case["layers"])}
    if kind == "qaoa":
        return {"bytes": 2.0 * item * 2.0 ** case["n"], "flops": _qaoa_flops(case["n"], case["p"])}
    if kind == "results":
        n = case["n"]
        # each term: a product and a sum of the amplitudes' pairs
        return {"bytes": item * 2.0 ** n + 8.0 * case["shots"], "flops": 4.0 * (4 * n - 3 + 6) * 2.0 ** n}
    if kind == "measure":
        # the state read, its surviving amplitudes written and read by the sampler
        return {"bytes": item * 2.0 ** case["n"] * (1.0 + 1.0 + 2.0 ** -case["m"]) + 8.0 * case["shots"],
                "flops": 10.0 * 2.0 ** case["n"]}
    if kind == "batch":
        mean = sum(2.0 ** n * n for n in range(case["n_min"], case["n_max"] + 1)) / (case["n_max"] - case["n_min"] + 1)
        states = sum(2.0 ** n for n in range(case["n_min"], case["n_max"] + 1)) / (case["n_max"] - case["n_min"] + 1)
        # 2.5 layers on average, 15 n operations a layer and amplitude
        return {"bytes": case["count"] * (2.0 * item * states + 96.0 * 100.0),
                "flops": case["count"] * 2.5 * 15.0 * mean}
    if kind == "noisy":
        n = case["n"]
        # the gates, and as many noise operators and their renormalisations again
        return {"bytes": case["trajectories"] * (8.0 + 2.0 * item * 2.0 ** n),
                "flops": case["trajectories"] * 3.0 * _layer_flops(n, case["layers"])}
    if kind == "serve":
        lo, hi = case["n_min"], case["n_max"]
        at = [int(lo * (hi / lo) ** (k / 64.0)) for k in range(64)]
        return {"bytes": case["requests"] * (sum(32.0 * 2.0 ** n for n in at) / 64 + 8.0 * case["shots"]),
                "flops": case["requests"] * sum(_layer_flops(n, 12) for n in at) / 64}
    n = case["n"]
    # one reduction to eigenvalues and vectors and one product: about 8 * (9 + 1) n^3 real operations
    return {"bytes": 32.0 * n * n, "flops": 80.0 * n ** 3}


# ---- the same outputs by plain torch / numpy in 64 bits -----------------------------
def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _zero_state(n: int):
    psi = torch.zeros(2 ** n, dtype=torch.complex128, device=_device())
    psi[0] = 1.0
    return psi


def _apply_1q(psi, n: int, q: int, m):
    v = psi.view(2 ** q, 2, -1)
    a = v[:, 0] * m[0][0] + v[:, 1] * m[0][1]
    b = v[:, 0] * m[1][0] + v[:, 1] * m[1][1]
    v[:, 0] = a
    v[:, 1] = b


def _cnot(psi, n: int, c: int, t: int):
    a, b = min(c, t), max(c, t)
    v = psi.view(2 ** a, 2, 2 ** (b - a - 1), 2, -1)
    on = v[:, 1] if c < t else v[:, :, :, 1]
    x, y = (on[:, :, 0], on[:, :, 1]) if c < t else (on[:, 0], on[:, 1])
    x2 = x.clone()
    x.copy_(y)
    y.copy_(x2)


def _exact_ops(n: int, ops):
    psi = _zero_state(n)
    r = math.sqrt(0.5)
    names = {v: k for k, v in _abi.OP.items()}
    for op in ops:
        k, q, h = names[int(op["kind"])], int(op["q"][0]), float(op["angle"]) / 2
        if k == "CNOT":
            _cnot(psi, n, q, int(op["q"][1]))
            continue
        c, s = math.cos(h), math.sin(h)
        m = {"H": [[r, r], [r, -r]], "RX": [[c, -1j * s], [-1j * s, c]], "RY": [[c, -s], [s, c]],
             "RZ": [[complex(c, -s), 0.0], [0.0, complex(c, s)]]}[k]
        _apply_1q(psi, n, q, m)
    return psi


def _exact_z(psi, n: int):
    p = psi.real ** 2 + psi.imag ** 2
    out = []
    for q in range(n):
        v = p.view(2 ** q, 2, -1)
        out.append(float(v[:, 0].sum() - v[:, 1].sum()))
    return np.array(out)


def _exact_zz(p, n: int, i: int, j: int) -> float:
    v = p.view(2 ** i, 2, 2 ** (j - i - 1), 2, -1)
    return float((v[:, 0, :, 0].sum() + v[:, 1, :, 1].sum()) - (v[:, 0, :, 1].sum() + v[:, 1, :, 0].sum()))


def _exact_qaoa(inst: dict):
    """The ansatz from its definition: phases of the whole cost function, then RX on every qubit."""
    n = inst["n"]
    x = torch.arange(2 ** n, dtype=torch.int64, device=_device())
    cost = torch.zeros(2 ** n, dtype=torch.float64, device=_device())
    for i, j, w in inst["graph"]:
        cost += -0.5 * w * (1.0 - 2.0 * (((x >> (n - 1 - i)) ^ (x >> (n - 1 - j))) & 1))
    psi = torch.full((2 ** n,), 2.0 ** (-n / 2), dtype=torch.complex128, device=_device())
    ps = inst["params"]
    for k in range(0, len(ps), 2):
        psi *= torch.polar(torch.ones_like(cost), -ps[k] * cost)
        c, s = math.cos(ps[k + 1]), math.sin(ps[k + 1])
        for q in range(n):
            _apply_1q(psi, n, q, [[c, -1j * s], [-1j * s, c]])
    return psi, cost


def _exact_pauli(psi, n: int, string: str) -> float:
    phi = psi.clone()
    mats = {"X": [[0, 1], [1, 0]], "Y": [[0, -1j], [1j, 0]], "Z": [[1, 0], [0, -1]]}
    for q, ch in enumerate(string):
        if ch != "I":
            _apply_1q(phi, n, q, mats[ch])
    return float(torch.vdot(psi, phi).real)


def exact(case: dict, seed: int):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    if kind == "layers":
        n = case["n"]
        psi = _exact_ops(n, workloads.random_layer_ops(n, case["layers"], seed))
        out = {"amplitudes": psi.cpu().numpy()} if n <= AMPLITUDES_UP_TO else {"z": _exact_z(psi, n)}
        if case["shots"]:
            out["shots"] = None
        return out
    if kind == "qaoa":
        inst = _qaoa(case["n"], case["p"], rng)
        psi, _ = _exact_qaoa(inst)
        p = psi.real ** 2 + psi.imag ** 2
        return {"zz": np.array([_exact_zz(p, case["n"], i, j) for i, j, _ in inst["graph"]])}
    if kind == "results":
        n = case["n"]
        psi = _exact_ops(n, workloads.random_layer_ops(n, 2, seed))
        one = []
        for q, m in _observables(n, rng):
            phi = psi.clone()
            _apply_1q(phi, n, q, m.tolist())
            one.append(complex(torch.vdot(psi, phi)))
        return {"shots": None, "terms": np.array([_exact_pauli(psi, n, s) for s in _chain_strings(n)]),
                "observables": np.array(one)}
    if kind == "measure":
        n = case["n"]
        psi = _exact_ops(n, workloads.random_layer_ops(n, 2, seed))
        p = (psi.real ** 2 + psi.imag ** 2).view([2] * n)
        qubits = sorted(int(q) for q in rng.choice(n, case["m"], replace=False))
        rest = [q for q in range(n) if q not in qubits]
        # outcome bit j is the j-th measured qubit: the last measured qubit varies slowest
        probs = p.sum(dim=rest) if rest else p
        return {"outcome": None, "probabilities": probs.permute(*reversed(range(case["m"]))).reshape(-1).cpu().numpy(),
                "shots": None}
    if kind == "batch":
        energies = []
        for inst in _batch_instances(case, seed):
            psi, cost = _exact_qaoa(inst)
            h = cost + sum(0.5 * w for _, _, w in inst["graph"])
            energies.append(((psi.real ** 2 + psi.imag ** 2) * h).sum())
        return {"energies": torch.stack(energies).cpu().numpy()}
    if kind == "expm":
        w, v = np.linalg.eigh(_hermitian(case["n"], seed))
        return {"exp": (v * np.exp(-1j * w)) @ v.conj().T}
    return None
