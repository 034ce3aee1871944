"""The single-pass scan resets its tile states in the launch that wrote them,
so a block may count itself finished only when its own stores to the states
have been performed.  No run shows a missing wait reliably; the compiled
kernels do."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "granular_gpu_amd" / "csrc"
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="no hipcc")
def test_scan_waits_for_its_state_stores_before_it_counts_itself(tmp_path):
    flags = subprocess.run(["make", "-s", "-C", str(CSRC), "--eval=flags:;@echo $(HIPFLAGS)",
                            "flags"], check=True, capture_output=True, text=True).stdout.split()
    out = tmp_path / "grid.s"
    subprocess.run([HIPCC, *flags, "--cuda-device-only", "-S", "grid.hip", "-o", str(out)],
                   cwd=CSRC, check=True, capture_output=True)
    bodies = re.findall(r"^_ZN2gg6k_scanILi\d+E.*?:\n(.*?)s_endpgm", out.read_text(), re.S | re.M)
    assert len(bodies) == 2  # both tile lengths
    for body in bodies:
        lines = [ln.split(";")[0].strip() for ln in body.splitlines()]
        # the finish counter is the last atomic with a result: sync[1]
        finish = max(k for k, ln in enumerate(lines) if ln.startswith("global_atomic_add"))
        assert "offset:4 sc0" in lines[finish]
        memory = max(k for k, ln in enumerate(lines[:finish])
                     if re.match(r"(global|flat|buffer|scratch)_", ln))
        waits = [ln for ln in lines[memory + 1:finish] if ln.startswith("s_waitcnt")]
        assert any("vmcnt(0)" in ln for ln in waits), lines[memory:finish + 1]
