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


@pytest.mark.gpu
def test_tensors_live_until_the_call_has_their_addresses(monkeypatch):
    """A library call gets addresses and releases the interpreter lock: every tensor behind them has to be alive then, or
    another thread may be handed its memory.  Looked at from inside the calls: no address of theirs is free memory."""
    import numpy as np

    from nl_hecate_amd import serving as SG
    from nl_hecate_amd.cms import ContextState, Pulse
    from nl_hecate_amd.ffi import lib
    from tests.test_gpu_serving import gpu_params
    from tests.test_oracle_serving import model

    def live(address):
        for seg in torch.cuda.memory_snapshot():
            at = seg["address"]
            if at <= address < at + seg["total_size"]:
                for block in seg["blocks"]:
                    if at <= address < at + block["size"]:
                        return block["state"] == "active_allocated"
                    at += block["size"]
        return True   # not of this allocator

    names = ("embedding_gather_cuda", "titans_forward_f32_cuda", "titans_final_states_f32_rocm")
    seen = []
    for name in names:
        def call(*args, fn=getattr(lib, name), name=name):
            seen.append(name)
            assert all(live(a) for a in args if isinstance(a, int) and a > 1 << 20), name
            return fn(*args)
        monkeypatch.setitem(lib.__dict__, name, call)
    nh, hd, v, s = 2, 32, 50, 40
    gp = gpu_params(model(nh * hd, v, 1, 3))
    memory = lambda: torch.zeros(nh, hd * hd, device="cuda")
    ML.gpu_memory_forward(gp.levels[0], ML.LevelConfig("titans", nh, hd), torch.randn(s, nh * hd, device="cuda"), memory(), s, nh * hd, 1)
    cfg = SG.ServeConfig(nh * hd, v, nh, hd, 16, s, [ML.LevelConfig("titans", nh, hd)], decode_tokens=2)
    SG.gpu_prefill_forward(gp, cfg, np.arange(s), Pulse(0, [True]), ContextState([memory()]))
    assert set(seen) == set(names)
