"""The compiled torch binding against the general path of beam/_C.py (torch_binding_check.py, in a process of its own)."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu


def test_binding_and_general_path_agree(gpu):
    script = os.path.join(os.path.dirname(os.path.abspath(__file__)), "torch_binding_check.py")
    r = subprocess.run([sys.executable, "-u", script], capture_output=True, text=True, timeout=110)
    assert r.returncode == 0 and "torch binding OK" in r.stdout, r.stdout[-3000:] + r.stderr[-3000:]
