"""Build libqsv.so in-tree with hipcc for gfx950.

    python -m qclojure_amd.build
"""
from __future__ import annotations

import os
import re
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT = os.path.join(HERE, "libqsv.so")
ARCH = os.environ.get("QSV_OFFLOAD_ARCH", "gfx950")

SOURCES = ["qsv_api.hip", "qsv_compile.hip", "qsv_gates.hip", "qsv_pass.hip", "qsv_small.hip", "qsv_kernels.hip", "qsv_pauli.hip", "qsv_batch.hip", "qsv_la.hip"]

HIPCC_FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
    # no packed-FP32 instructions in device code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-result", "-Wno-unused-value",
]
# The files that run micro-op programs:
_OPS_FLAGS = [
    # uniform branches stay branches: structurised, the op dispatch of a fused
    # pass keeps a second copy of the tile in registers (128 VGPRs and 2500
    # spills instead of 101 and none). No vector combining: it turns a slot's
    # scalar into a two-slot vector load, which keeps FP32 tiles in scratch.
    "-mllvm", "-structurizecfg-skip-uniform-regions=true", "-mllvm", "-disable-vector-combine",
    # both are the compiler's internals: what its kernels take is checked (spills)
    "-Rpass-analysis=kernel-resource-usage",
]
FILE_FLAGS = {"qsv_pass.hip": _OPS_FLAGS, "qsv_small.hip": _OPS_FLAGS}


def _noise(text: str) -> list[str]:
    out, remark = [], False
    for l in text.splitlines():
        if ": remark: " in l:
            remark = True   # the source lines that it quotes follow
        elif re.search(r": (warning|error|note): ", l):
            remark = False
        if l.strip() and not remark and "packed-fp32-ops" not in l and "not a recognized feature" not in l:
            out.append(l)
    return out


def spills(text: str) -> dict[str, tuple[int, int]]:
    """Scratch bytes a lane and spilled vector registers of every kernel in the compiler's resource remarks."""
    out: dict[str, tuple[int, int]] = {}
    name, scratch = None, 0
    for l in text.splitlines():
        m = re.search(r"remark: .*?(Function Name|ScratchSize \[bytes/lane\]|VGPRs Spill): (\S+)", l)
        if not m:
            continue
        if m[1] == "Function Name":
            name, scratch = m[2], 0
        elif m[1].startswith("Scratch"):
            scratch = int(m[2])
        elif name:
            out[name] = (scratch, int(m[2]))
    return out


def command(src: str, obj: str) -> list[str]:
    return ["hipcc", *HIPCC_FLAGS, *FILE_FLAGS.get(os.path.basename(src), []), "-c", "-o", obj, src]


def _compile(src: str, obj: str, verbose: bool) -> None:
    cmd = command(src, obj)
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError(f"hipcc failed on {src}")
    for kernel, (scratch, regs) in spills(r.stderr).items():
        if scratch or regs:
            sys.stderr.write(f"{os.path.basename(src)}: {kernel} keeps {scratch} bytes a lane in scratch "
                             f"({regs} spilled registers): this compiler does not honour the flags\n")
    if verbose and _noise(r.stdout + r.stderr):
        print("\n".join(_noise(r.stdout + r.stderr)))


def build(verbose: bool = False) -> str:
    srcs = [os.path.join(CSRC, s) for s in SOURCES if os.path.exists(os.path.join(CSRC, s))]
    tmp = OUT + ".tmp"
    with tempfile.TemporaryDirectory() as d:
        objs = [os.path.join(d, os.path.basename(s) + ".o") for s in srcs]
        with ThreadPoolExecutor(max(1, min(len(srcs), os.cpu_count() or 1, 8))) as ex:
            list(ex.map(lambda so: _compile(*so, verbose), zip(srcs, objs)))
        cmd = ["hipcc", f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            sys.stderr.write(r.stdout + r.stderr)
            raise RuntimeError("hipcc failed linking libqsv.so")
    os.replace(tmp, OUT)
    return OUT


if __name__ == "__main__":
    print(build(verbose=True))
