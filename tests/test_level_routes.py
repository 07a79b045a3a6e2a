"""Which levels may run as a batch: the grouped kernels take raw addresses, so whatever a call by name would refuse, and
whatever has another shape, type or layout than they read, has to go the level's own way."""
import dataclasses

import pytest
import torch

from nl_hecate_amd import memory_level as ML
from nl_hecate_amd.mag_layer import MemoryLevelParams

D, NH = 64, 2


def params(device, **change):
    z = lambda *sh: torch.zeros(*sh, device=device)
    p = MemoryLevelParams(z(D, D), z(D, D), z(D, D), z(2 * D), z(1), z(2 * D), z(1), z(2 * D), z(1))
    return dataclasses.replace(p, **change)


def key(p, rule="titans"):
    return ML.group_key(ML.LevelConfig(rule, NH, D // NH), p, D, 1)


def test_host_tensors_have_no_key():
    assert key(params("cpu")) is None
    assert not ML._plain(torch.zeros(4)) and not ML._plain(None)


@pytest.mark.gpu
def test_keys_of_device_tensors():
    assert key(params("cuda")) is not None and key(params("cuda")) == key(params("cuda"))
    # the momentum gate's tensors are not looked at without momentum
    assert key(params("cuda", w_eta=None, b_eta=None), "delta") is not None
    assert key(params("cuda", w_eta=None), "titans") is None


@pytest.mark.gpu
@pytest.mark.parametrize("name", [f.name for f in dataclasses.fields(MemoryLevelParams)])
def test_no_key_with_one_tensor_that_the_kernels_cannot_read(name):
    good = getattr(params("cuda"), name)
    bad = [good.cpu(), good.double(), good.to(torch.bfloat16), good[:0]]
    if good.numel() > 1:
        bad.append(good[:D // 2].contiguous() if good.dim() == 1 else good[:D // 2])
        bad.append(torch.zeros(good.numel() + 1, device="cuda")[1:].view(good.shape))                   # 4 bytes off
        bad.append(good.t() if good.dim() == 2 and good.t().is_contiguous() is False else good[::2])
    for t in bad:
        assert key(params("cuda", **{name: t})) is None, (name, t.shape, t.dtype, t.device)


@pytest.mark.gpu
def test_gradient_buffers_that_the_grouped_backward_writes():
    assert ML._grads_plain(ML.LevelGrads.zeros(D), D)
    for name, t in (("d_w_k_mem", torch.zeros(D, D)), ("d_w_q_mem", torch.zeros(D, D, device="cuda", dtype=torch.float64)),
                    ("d_w_v_mem", torch.zeros(D // 2, D, device="cuda")), ("d_w_alpha", torch.zeros(D, device="cuda")),
                    ("d_b_theta", torch.zeros(1)), ("d_w_eta", None)):
        assert not ML._grads_plain(dataclasses.replace(ML.LevelGrads.zeros(D), **{name: t}), D), name
