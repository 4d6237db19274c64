"""The compiled torch binding only makes calls cheaper: the library builds without torch, and the package works without the binding."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "general-nvgpu-testing_amd")


def plan(python):
    return subprocess.run(["make", "-n", "-B", "-C", os.path.join(PKG, "csrc"), "all", f"PYTHON={python}"], capture_output=True, text=True)


def test_library_builds_without_torch():
    without = plan(f"{sys.executable} -S")  # sees no installed package
    assert without.returncode == 0, without.stderr
    assert "libbeam_hip.so" in without.stdout and "torch" not in without.stdout and not without.stderr, without.stderr
    assert "-o ../beam/_torch_binding.so" in plan(sys.executable).stdout


def imported(before):
    code = f"import sys\nsys.path.insert(0, {PKG!r})\nimport torch\n{before}\nimport beam\nfrom beam import _C\nprint('native:', _C._native)\n"
    return subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300)


def test_import_without_the_binding():
    r = imported("sys.modules['beam._torch_binding'] = None  # the import of it fails")
    assert r.returncode == 0 and "native: None" in r.stdout, r.stderr
    assert r.stderr.count("RuntimeWarning") == 1, r.stderr
    r = imported("")
    assert r.returncode == 0 and "_torch_binding.so" in r.stdout and "RuntimeWarning" not in r.stderr, r.stderr
