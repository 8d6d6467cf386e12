"""The kernels that run micro-op programs hold their tile in registers: the
compiler's own account of a build says that none of them spills."""
from __future__ import annotations

import os
import shutil
import subprocess

import pytest

from qclojure_amd import build


def test_remarks_are_read():
    text = "\n".join(f"a.hip:1:0: remark: {l} [-Rpass-analysis=kernel-resource-usage]" for l in (
        "Function Name: k_one", "    VGPRs: 101", "    ScratchSize [bytes/lane]: 0", "    SGPRs Spill: 10",
        "    VGPRs Spill: 0", "Function Name: k_two", "    ScratchSize [bytes/lane]: 212", "    VGPRs Spill: 53"))
    assert build.spills(text) == {"k_one": (0, 0), "k_two": (212, 53)}
    assert build._noise(text + "\n   1 | quoted\nb.hip:2:1: warning: unused\n") == ["b.hip:2:1: warning: unused"]


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="no hipcc")
def test_fused_passes_do_not_spill(tmp_path):
    src = os.path.join(build.CSRC, "qsv_pass.hip")
    cmd = build.command(src, str(tmp_path / "pass.o"))
    r = subprocess.run([cmd[0], "--cuda-device-only", *cmd[1:]], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    found = build.spills(r.stderr)
    assert sum("k_pass" in k for k in found) >= 5   # both precisions, with and without the norm
    assert all(v == (0, 0) for v in found.values()), found
