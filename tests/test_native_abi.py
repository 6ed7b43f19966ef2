"""CPU: the native dispatch refuses a library of another ABI version.

The extension resolves the library's functions by name, so a library from another build would be
called with other arguments. A stub that claims an older version is put before the real library in
the dynamic linker's order, in a process of its own."""
from __future__ import annotations

import shutil
import subprocess
import sys
from pathlib import Path

import pytest

from sihc_hip import _lib, _native

PROGRAM = """
import ctypes, sys
sys.path.insert(0, {package!r})
import torch
ctypes.CDLL({stub!r}, mode=ctypes.RTLD_GLOBAL)
import importlib.util
spec = importlib.util.spec_from_file_location("_sihc_torch", {native!r})
try:
    importlib.util.module_from_spec(spec)
except ImportError as e:
    print("refused:", e)
else:
    print("loaded")
"""


@pytest.mark.parametrize("shift", [0, -1])
def test_the_extension_checks_the_library_version(tmp_path, shift):
    source, stub = tmp_path / "stub.c", tmp_path / "stub.so"
    source.write_text(f"int sihc_abi_version(void) {{ return {_lib.ABI_VERSION + shift}; }}\n")
    subprocess.run([shutil.which("gcc") or "cc", "-shared", "-fPIC", "-o", str(stub), str(source)], check=True)
    program = PROGRAM.format(package=str(Path(_lib.__file__).parents[1]), stub=str(stub), native=str(_native.NATIVE_PATH))
    out = subprocess.run([sys.executable, "-c", program], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stderr
    if shift:
        assert out.stdout.startswith("refused:") and "rebuild" in out.stdout
    else:
        assert out.stdout.strip() == "loaded"


def test_the_module_loads_the_checked_library_first(monkeypatch):
    monkeypatch.setattr(_native, "_module", None)
    monkeypatch.setattr(_native, "lib", lambda: (_ for _ in ()).throw(RuntimeError("stale library")))
    with pytest.raises(RuntimeError, match="stale library"):
        _native.module()
