"""Checks of the Python layer that keep a wrong call from reaching a kernel; no GPU needed."""

import pytest
import torch

from xlb_amd import _lib


def test_a_host_tensor_has_no_stream():
    """The entry points that take raw pointers ask for the tensor's stream: one that is not on a GPU
    is refused there, whatever device is current."""
    with pytest.raises(ValueError, match="GPU"):
        _lib.stream_of(torch.zeros(3))
