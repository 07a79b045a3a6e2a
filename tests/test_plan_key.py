"""The key that an argument block of tensor addresses is kept under: whatever a tensor can change where it stands shows."""
import importlib.util
import os
import subprocess

import numpy as np
import pytest
import torch

from nl_hecate_amd import ffi

if not os.path.exists(ffi.KEY_PATH):   # host code: builds without the library
    subprocess.check_call(["make", "-s", "-C", os.path.join(os.path.dirname(os.path.abspath(ffi.__file__)), "csrc"), "plan_key"])


@pytest.fixture(params=["extension", "python"])
def tensor_key(request, monkeypatch, tmp_path):
    """The key by the extension, and where it was not built."""
    if request.param == "extension":
        return lambda tensors: ffi.tensor_key(tensors)
    fresh = importlib.util.module_from_spec(importlib.util.find_spec("nl_hecate_amd.ffi"))   # nothing loaded yet
    fresh.__loader__.exec_module(fresh)
    monkeypatch.setattr(fresh, "KEY_PATH", str(tmp_path / "plan_key.so"))
    with pytest.warns(UserWarning, match="cannot be loaded"):
        fresh.tensor_key([])
    return lambda tensors: fresh.tensor_key(tensors)


@pytest.mark.parametrize("change", ["nothing", "values", "transpose", "shape", "resize", "data", "type", "view"])
def test_key_of_a_tensor_that_changed_where_it_stands(change, tensor_key):
    t, other = torch.zeros(6, 6), torch.zeros(2, 3, dtype=torch.bfloat16)
    before = tensor_key([t, other])
    assert isinstance(before, bytes) and before == tensor_key((t, other))
    keep = t.data
    if change == "values":
        t.add_(1)
    elif change == "transpose":
        t.t_()
    elif change == "shape":
        t.data = keep.view(36)
    elif change == "resize":
        t.resize_(6, 5)
    elif change == "data":
        t.data = torch.zeros(6, 6)
    elif change == "type":
        t.data = keep.view(torch.int32)
    elif change == "view":
        t = t[1:]
    assert (before == tensor_key([t, other])) == (change in ("nothing", "values"))


@pytest.mark.parametrize("shape", [(), (4,), (2, 3), (2, 0, 5)])
def test_key_says_how_many_sizes_follow(shape):
    """Type, device and rank share a word; the -1 that stands for the device index of a CPU tensor is not to cover the rank."""
    words = np.frombuffer(ffi.tensor_key([torch.zeros(shape)]), np.int64)
    assert len(words) == 2 + 2 * len(shape) and words[1] >> 32 == len(shape)


def test_key_of_what_has_no_address(tensor_key):
    assert tensor_key([]) == b""
    for bad, error in (([None], TypeError), ([1.0], TypeError), (3, TypeError),
                       ([torch.zeros(2, device="meta"), "w"], TypeError)):
        with pytest.raises(error):
            tensor_key(bad)
    sparse = torch.eye(3).to_sparse()
    with pytest.raises(RuntimeError):
        tensor_key([sparse])
