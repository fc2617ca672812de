"""The native argument checks are optional: a build of them that this Python or
torch cannot use is left aside with one warning, at the first call and at every
later one alike, and libtq4.so builds without torch or Python."""
import os
import shutil
import subprocess
import sys
import sysconfig

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(REPO, "ascend-micro-harness_amd")
EXT = "_tq4_host" + sysconfig.get_config_var("EXT_SUFFIX")

PROGRAM = """
import importlib, sys, warnings
import torch
if {version!r}:
    torch.__version__ = {version!r}
sys.path.insert(0, {root!r})
tq4 = importlib.import_module("pkg.tq4")
with warnings.catch_warnings(record=True) as seen:
    warnings.simplefilter("always")
    for _ in range(3):
        assert tq4.status_string(0) == "ok"
        assert tq4.auto_splits(1, 8, 256, 16) == 16
print(tq4._fast is not None, [str(w.message) for w in seen if w.category is RuntimeWarning])
"""


def run(tmp_path, host, version=None):
    root = tmp_path / "pkg"
    root.mkdir()
    for f in ("tq4.py", "libtq4.so"):
        shutil.copy(os.path.join(PKG, f), root)
    (root / "__init__.py").write_text("")
    if host is not None:
        (root / EXT).write_bytes(host)
    r = subprocess.run([sys.executable, "-c", PROGRAM.format(root=str(tmp_path), version=version)],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    used, messages = r.stdout.strip().splitlines()[-1].split(" ", 1)
    return used == "True", messages


@pytest.fixture(scope="module")
def built():
    path = os.path.join(PKG, EXT)
    if not os.path.exists(path):
        pytest.skip(f"{EXT} is not built (make -C ascend-micro-harness_amd/csrc host)")
    with open(path, "rb") as f:
        return f.read()


def test_used_as_built(tmp_path, built):
    assert run(tmp_path, built) == (True, "[]")


def test_absent(tmp_path):
    assert run(tmp_path, None) == (False, "[]")


def test_not_loadable(tmp_path):
    used, messages = run(tmp_path, b"no shared object")
    assert not used and messages.count("_tq4_host is not used") == 1


def test_built_for_another_torch(tmp_path, built):
    used, messages = run(tmp_path, built, version="0.1.0+rocm")
    assert not used and messages.count("_tq4_host is not used") == 1


def test_default_target_needs_hipcc_alone():
    r = subprocess.run(["make", "-n", "-B", "-C", os.path.join(PKG, "csrc"), "PYTHON=/nonexistent"],
                       capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "nonexistent" not in r.stderr, r.stderr
    assert "libtq4.so" in r.stdout and "tq4_host" not in r.stdout and "python" not in r.stdout
