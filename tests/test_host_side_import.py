"""The package without its C++ host side (_torch_calls): calls run the Python
host side, whether the extension is missing or cannot be loaded, and the
errors of a missing kernel library stay the library's.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                   "tpu-native-pallas-flashattention_amd", "pallas_flash")
EXT = "_torch_calls" + sysconfig.get_config_var("EXT_SUFFIX")

PROGRAM = """
import warnings, torch
import pallas_flash as pf
from pallas_flash import _lib
x = torch.zeros(1, 2, 4, 64)
with warnings.catch_warnings(record=True) as seen:
    warnings.simplefilter("always")
    for call in (lambda: pf.flash_attention(x, x, x, kv_len=0), lambda: pf.flash_attention(x, x, x),
                 lambda: pf.flash_attention_decode(x[:, :, :1], x, x, 3)):
        try:
            call()
        except Exception as e:
            print(type(e).__name__, str(e)[:60])
print("warned", sum("host side" in str(w.message) for w in seen), "native", hasattr(_lib.calls(), "__file__"))
try:
    _lib.lib()
except RuntimeError as e:
    print(e)
"""


def _run(tmp_path, ext, lib=True):
    pkg = tmp_path / "pallas_flash"
    pkg.mkdir()
    for f in os.listdir(PKG):
        if f.endswith(".py"):
            shutil.copy(os.path.join(PKG, f), pkg)
    if lib:
        os.symlink(os.path.join(PKG, "libpallas_flash_amd.so"), pkg / "libpallas_flash_amd.so")
    if ext is not None:
        (pkg / EXT).write_bytes(ext)
    r = subprocess.run([sys.executable, "-c", PROGRAM], cwd=tmp_path, capture_output=True, text=True, timeout=300,
                       env={**os.environ, "PYTHONPATH": str(tmp_path)})
    assert r.returncode == 0, r.stderr
    return r.stdout


@pytest.mark.parametrize("ext", [None, b"of another system"])
def test_calls_run_without_the_extension(tmp_path, ext):
    out = _run(tmp_path, ext)
    assert "ValueError kv_len must be in" in out  # the general path's own checks
    assert out.count("RuntimeError pallas_flash (MI355X) runs its HIP kernels") == 2  # CPU tensors
    assert "warned 1 native False" in out


def test_arguments_are_checked_without_the_library(tmp_path):
    out = _run(tmp_path, None, lib=False)
    assert "ValueError kv_len must be in" in out and "warned 0" in out
    assert "libpallas_flash_amd.so is not built" in out


def test_the_extension_is_the_one_of_this_python_and_torch():
    from pallas_flash import _lib
    assert os.path.basename(_lib.calls().__file__) == EXT
