import ctypes
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
for p in (ROOT, ROOT / "oracle"):
    if str(p) not in sys.path:
        sys.path.insert(0, str(p))


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP path)")


@pytest.fixture(scope="session")
def gpu(tmp_path_factory):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.init()
    # a process that dies in native code names the place
    so = tmp_path_factory.mktemp("native") / "native_trace.so"
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", str(ROOT / "tests" / "native_trace.c"), "-o", str(so)],
                   check=True)
    ctypes.CDLL(str(so)).native_trace()
    return torch.device("cuda:0")
