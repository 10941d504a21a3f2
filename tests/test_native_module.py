"""CPU checks of how the native module is found: the package imports and the
library loads without it, with one that does not load, and with one built for
another torch (the calls then go through ctypes)."""
import os
import shutil
import subprocess
import sys

import pytest
import torch

from mlxcel_amd import _lib, ops

pytestmark = pytest.mark.skipif(not os.path.exists(_lib.LIB_PATH), reason="library not built here")

CHECK = """
import warnings
with warnings.catch_warnings(record=True) as seen:
    warnings.simplefilter("always")
    import mlxcel_amd
    from mlxcel_amd import _lib, ops
print(_lib.load().mlxq_version().decode())
print("ctypes" if ops._native is ops._ctypes_only else "native", len([w for w in seen if "ctypes" in str(w.message)]))
"""


@pytest.mark.parametrize("module", ["missing", "broken", "no library", "as built"])
def test_import_and_load(tmp_path, module):
    pkg = tmp_path / "mlxcel_amd"
    pkg.mkdir()
    here = os.path.dirname(_lib.__file__)
    for f in os.listdir(here):
        if f.endswith(".py"):
            shutil.copy(os.path.join(here, f), pkg)
    if module != "no library":
        os.symlink(_lib.LIB_PATH, pkg / "libmlxq.so")
    if module == "broken":
        (pkg / "_mlxq_native.so").write_bytes(b"not a shared object")
    elif module != "missing":
        if not os.path.exists(_lib.NATIVE_PATH):
            pytest.skip("native module not built here")
        shutil.copy(_lib.NATIVE_PATH, pkg)
    r = subprocess.run([sys.executable, "-c", CHECK], cwd=tmp_path, capture_output=True, text=True,
                       env={**os.environ, "PYTHONPATH": str(tmp_path)})
    if module == "no library":  # the import goes through, load() says what is missing
        assert "LibraryNotBuilt" in r.stderr, r.stderr
        return
    assert r.returncode == 0, r.stderr
    how = {"missing": "ctypes 0", "broken": "ctypes 1", "as built": "native 0"}[module]
    assert r.stdout.split("\n")[1] == how, r.stdout


def test_a_module_for_another_torch_is_not_used(monkeypatch):
    if ops._native is ops._ctypes_only:
        pytest.skip("native module not built here")
    monkeypatch.setattr(torch, "__version__", "0.0.1")
    with pytest.warns(UserWarning, match="built for torch"):
        assert ops._load_native() is ops._ctypes_only
