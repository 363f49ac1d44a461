"""Checks of the Python layer that keep a wrong call from reaching a kernel; no GPU needed."""

import subprocess

import pytest
import torch

from xlb_amd import _lib


def test_a_host_tensor_has_no_stream():
    """The entry points that take raw pointers ask for the tensor's stream: one that is not on a GPU
    is refused there, whatever device is current."""
    with pytest.raises(ValueError, match="GPU"):
        _lib.stream_of(torch.zeros(3))


def test_a_library_of_another_version_is_named_as_such(tmp_path, monkeypatch):
    """A library built from older sources lacks entries that this package binds: the error is about
    its version, not about the first missing symbol."""
    source, old = tmp_path / "old.c", tmp_path / "libold.so"
    source.write_text("int xlbh_abi_version(void) { return 4; }\n")
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(old), str(source)], check=True)
    monkeypatch.setattr(_lib, "LIB_PATH", str(old))
    monkeypatch.setattr(_lib, "_LIB", None)
    with pytest.raises(RuntimeError, match="ABI version 4"):
        _lib.lib()
