"""A library of the bindings' version from before an entry point was added."""
import subprocess

import pytest


def test_a_library_without_an_entry_point_asks_for_a_rebuild(pkg, monkeypatch, tmp_path):
    lib = pkg._lib
    src = tmp_path / "old.c"
    src.write_text(f"int svbrdf_abi_version(void) {{ return {lib.ABI_VERSION}; }}\n")
    so = tmp_path / "old.so"
    subprocess.run(["gcc", "-shared", "-fPIC", str(src), "-o", str(so)], check=True)
    monkeypatch.setattr(lib, "LIB_PATH", so)
    monkeypatch.setattr(lib, "_lib", None)
    with pytest.raises(ImportError, match="rebuild"):
        lib.load()
    assert lib._lib is None
