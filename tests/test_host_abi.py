"""A library or a host module left from another build is refused with TileMixLibraryError, before
anything is bound or called (CPU)."""
from __future__ import annotations

import shutil
import subprocess
import types

import pytest

from tilemix_amd import _native


def _library(tmp_path, name, source):
    src, out = tmp_path / f"{name}.c", tmp_path / f"{name}.so"
    src.write_text(source)
    subprocess.run([shutil.which("gcc") or "cc", "-shared", "-fPIC", str(src), "-o", str(out)], check=True)
    return out


def test_library_of_another_version(tmp_path):
    """The version is asked before any symbol that such a library may not have."""
    old = _library(tmp_path, "old", "int tilemix_abi_version(void) { return 3; }\n")
    with pytest.raises(_native.TileMixLibraryError, match="ABI version 3 != "):
        _native.load_library(old)
    with pytest.raises(_native.TileMixLibraryError, match="no tilemix_abi_version"):
        _native.load_library(_library(tmp_path, "none", "int other(void) { return 0; }\n"))
    short = _library(tmp_path, "short", "int tilemix_abi_version(void) { return %d; }\n" % _native.ABI_VERSION)
    with pytest.raises(_native.TileMixLibraryError, match="does not export .*tilemix_attn_fwd_uniform"):
        _native.load_library(short)


def test_host_module_matches_what_is_loaded():
    lib = _native.load_library()
    _native.host()  # the built one passes
    abi, sizes, torch_id = __import__("tilemix_amd._host", fromlist=["built_for"]).built_for()
    assert abi == _native.ABI_VERSION and len(sizes) == 4
    for stale in ((abi - 1, sizes, torch_id), (abi, (sizes[0], sizes[1] + 8, *sizes[2:]), torch_id),
                  (abi, sizes, "2.9.0 0123")):
        with pytest.raises(_native.TileMixLibraryError, match="_host.so was built for"):
            _native._check_host(types.SimpleNamespace(built_for=lambda: stale), lib)
    with pytest.raises(_native.TileMixLibraryError, match="_host.so was built for None"):
        _native._check_host(types.SimpleNamespace(), lib)
