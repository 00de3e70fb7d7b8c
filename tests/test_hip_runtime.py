"""One HIP runtime per process, whichever of torch and the runtime library is
loaded first (each would bring its own copy). Loads libraries only: no GPU."""
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
TORCH = "import torch"
OURS = "from rtlflow_amd.model import runtime; runtime()"
MAPS = """
import re
hip = {ln.split()[-1] for ln in open("/proc/self/maps") if re.search(r"/lib(amdhip64|hsa-runtime64)[.]so", ln)}
print("\\n".join(sorted(hip)))
"""


@pytest.mark.parametrize("order", [(OURS,), (TORCH, OURS), (OURS, TORCH)])
def test_one_hip_runtime_in_either_order(order):
    code = "\n".join(order) + MAPS
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    libs = r.stdout.split()
    assert len([p for p in libs if "libamdhip64" in p]) == 1, libs
    assert len([p for p in libs if "libhsa-runtime64" in p]) == 1, libs


STREAM = """
from rtlflow_amd.designs import registry
from rtlflow_amd.model import MODE_FUSED
cd = registry.get("net_tiny")              # loads the runtime
import torch
with cd.model(64) as m:
    nin, _ = m.stream_words()
    x = torch.zeros((5, nin, 64), dtype=torch.int64, device="cuda")
    m.set_input_stream(x)
    m.begin(1)
    m.run_cycles(5, MODE_FUSED)
    got = m.hashes()
    assert len(set(got.tolist())) == 1, got
print("STREAM OK", flush=True)
"""


@pytest.mark.gpu
def test_torch_buffers_are_known_when_the_runtime_comes_first(gpu):
    """A model whose library was loaded before torch takes a torch tensor as
    its input stream (all-zero inputs: every stimulus hashes alike)."""
    r = subprocess.run([sys.executable, "-u", "-c", STREAM], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "STREAM OK" in r.stdout, r.stdout[-1000:] + r.stderr[-2000:]
