"""Loading a library that does not belong to the binding (an older tree's, or of another
ABI version) says so and asks for a rebuild, whatever it lacks."""
import os
import shutil
import subprocess

import pytest

from botorch_amd import _lib

CC = shutil.which("gcc") or shutil.which("cc")


@pytest.mark.skipif(CC is None, reason="no C compiler")
@pytest.mark.parametrize("source", [
    "int unrelated(void) { return 0; }",
    "int bta_abi_version(void) { return %d; }" % (_lib.ABI_VERSION - 1),
    "int bta_abi_version(void) { return %d; }\n"
    "const char* bta_version(void) { return 0; }" % _lib.ABI_VERSION])
def test_a_library_of_another_tree_asks_for_a_rebuild(tmp_path, monkeypatch, source):
    src, so = tmp_path / "other.c", tmp_path / "libother.so"
    src.write_text(source)
    subprocess.run([CC, "-shared", "-fPIC", "-o", str(so), str(src)], check=True, timeout=60)
    monkeypatch.setattr(_lib, "_lib", None)
    with pytest.raises(RuntimeError, match="rebuild the library"):
        _lib.load(str(so))
    assert _lib._lib is None
    assert os.path.exists(_lib.LIB_PATH) and _lib.load() is not None
