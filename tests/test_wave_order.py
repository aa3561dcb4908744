"""LDS data handed between lanes of one wave is ordered in the program, not
only in the instructions that a compiler happened to choose: in the optimized
LLVM IR of a kernel that does so, a fence stands between every store to LDS
and the load after it, and between every load and the store after it.
"""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "super-gemma_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def _lds_events(body):
    """The kernel's LDS stores (S), loads (L) and fences (F) in program text order."""
    events = []
    for line in body.splitlines():
        if re.search(r"\bfence\b.*(acquire|release|acq_rel|seq_cst)", line):
            events.append("F")
        elif re.search(r"\bstore\b.*ptr addrspace\(3\)", line):
            events.append("S")
        elif re.search(r"\bload\b.*ptr addrspace\(3\)", line):
            events.append("L")
    return events


@pytest.mark.skipif(not shutil.which(HIPCC), reason="no hipcc")
@pytest.mark.parametrize("source,kernel,count", [("mmq.hip", "mmq_skinny_kernel", 16)])
def test_lds_exchanges_within_a_wave_are_fenced(tmp_path, source, kernel, count):
    out = tmp_path / "device.ll"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", "--offload-device-only", "-emit-llvm", "-S",
                    os.path.join(CSRC, source), "-o", str(out)],
                   check=True, capture_output=True)
    found = re.findall(r"^define [^\n]*@(\w*%s\w*)\([^\n]*\{\n(.*?)^\}" % kernel, out.read_text(),
                       re.S | re.M)
    assert len(found) == count
    for name, body in found:
        events = "".join(_lds_events(body))
        assert "S" in events and "L" in events
        assert "SL" not in events and "LS" not in events, (name, events)
