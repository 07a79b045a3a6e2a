"""The forwards of the exact and frozen rules run with and without scratch memory: a cold call under capture and calls on a
second stream walk the tokens, as they did before they had a form that wants scratch; long sequences go through a bounded
amount of it in stretches; the state after the last token needs none."""
import ctypes

import numpy as np
import pytest
import torch

from nl_hecate_amd import dispatch as D
from nl_hecate_amd.ffi import lib
from oracle import pyoracle as orc
from tests.gpu_util import assert_close, dev, host, rule_inputs
from tests.test_gpu_exact_mm import F32_MAX, kernels_run

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def empty_workspace():
    lib.nlh_release_workspace()
    yield
    lib.nlh_set_stream(None)
    lib.nlh_exact_backward_form(0)
    lib.nlh_release_workspace()


def forward(d=64, B=4, s=1000, C=64, seed=3):
    """-> (call, its outputs): shapes at which the matrix form is chosen."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    n = lambda *sh: torch.randn(*sh, generator=g, device="cuda")
    unit = lambda x: x / x.norm(dim=-1, keepdim=True)
    slots = -(-s // C) + 1
    x = [unit(n(B, s, d)), n(B, s, d), unit(n(B, s, d)), *(torch.sigmoid(n(B, s)) for _ in range(3)), 0.1 * n(B, d, d), 0.1 * n(B, d, d)]
    out = [torch.zeros(B, slots, d, d, device="cuda"), torch.zeros(B, slots, d, d, device="cuda"), torch.zeros(B, s, d, device="cuda")]
    return (lambda: D.call("titans_forward_ckpt_batched_f32_rocm", *x, *out, s, d, B, C, 0.0, F32_MAX)), out


def walk(call, out):
    lib.nlh_exact_backward_form(2)
    call()
    lib.nlh_exact_backward_form(0)
    torch.cuda.synchronize()
    return [host(t) for t in out]


def test_cold_capture_walks_the_tokens():
    call, out = forward()
    want = walk(call, out)
    for t in out:
        t.zero_()
    lib.nlh_release_workspace()
    torch.cuda.synchronize()
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=side):
        lib.nlh_set_stream(ctypes.c_void_p(side.cuda_stream))
        call()
        lib.nlh_set_stream(None)
    for i in range(3):
        for t in out:
            t.fill_(float(i))
        graph.replay()
        torch.cuda.synchronize()
        for t, w in zip(out, want):
            assert np.array_equal(host(t), w)
        assert "ex_scan_kernel" in kernels_run(call)   # eager work in between has its scratch
    # warm: the buffer that stands now is no part of a graph either
    warm = torch.cuda.CUDAGraph()
    with torch.cuda.graph(warm, stream=side):
        lib.nlh_set_stream(ctypes.c_void_p(side.cuda_stream))
        call()
        lib.nlh_set_stream(None)
    lib.nlh_release_workspace()
    warm.replay()
    torch.cuda.synchronize()
    for t, w in zip(out, want):
        assert np.array_equal(host(t), w)


def test_a_second_stream_does_not_share_the_scratch():
    (a, out_a), (b, out_b) = forward(seed=3), forward(seed=4)
    want = walk(b, out_b)
    assert "ex_scan_kernel" in kernels_run(a)
    first = [host(t) for t in out_a]
    side = torch.cuda.Stream()

    def both():
        for _ in range(4):
            lib.nlh_set_stream(ctypes.c_void_p(side.cuda_stream))
            b()
            lib.nlh_set_stream(None)
            a()
        torch.cuda.synchronize()

    both()
    for t, w in zip(out_b, want):
        assert np.array_equal(host(t), w)
    for t, w in zip(out_a, first):
        assert np.array_equal(host(t), w)
    lib.nlh_set_stream(ctypes.c_void_p(side.cuda_stream))
    ran = kernels_run(b)
    assert "rule_fwd_kernel" in ran and "ex_scan_kernel" not in ran
    lib.nlh_release_workspace()   # the next caller is the first again
    assert "ex_scan_kernel" in kernels_run(b)


@pytest.mark.parametrize("d,B,s", [(64, 80, 4 * 2180 + 3), (32, 640, 1500)])
def test_long_sequences_in_stretches(d, B, s):
    """More chunk maps than the scratch holds at once: 34 and 17 chunks of every chain to a stretch."""
    call, out = forward(d, B, s)
    want = walk(call, out)
    for t in out:
        t.zero_()
    lib.nlh_exact_backward_form(1)
    ran = kernels_run(call)
    lib.nlh_exact_backward_form(0)
    assert "ex_scan_kernel" in ran
    for t, w in zip(out, want):
        got = host(t)
        # both sides are within 1e-6 of the exact values (2-norms, tests of either form's rounding)
        assert np.linalg.norm((got - w).astype(np.float64)) <= 2e-6 * np.linalg.norm(w.astype(np.float64))


@pytest.mark.parametrize("rule", ["titans", "delta"])
@pytest.mark.parametrize("d", [8, 16, 32, 48, 64, 128])
@pytest.mark.parametrize("B,s", [(3, 1), (2, 15), (1, 16), (3, 130)])
def test_state_after_the_last_token(rule, d, B, s):
    x = rule_inputs(B, s, d, seed=5 + s + d, m0_scale=0.3)
    t = {n: dev(a) for n, a in x.items()}
    gates = [t[n] for n in (("alpha", "theta", "eta") if rule == "titans" else ("alpha", "theta"))]
    zero = np.zeros((d, d), np.float32)
    for form in (2, 1):      # the walk, in place; the matrix form where it exists
        lib.nlh_exact_backward_form(form)
        m = t["m0"].clone().view(B, d * d)
        args = [t["k"], t["v"], *gates, m] + ([None] if rule == "titans" else []) + [m, s, d, B]
        D.call(f"{rule}_final_states_f32_rocm", *args)
        for b in range(B):
            a = [x[n][b] for n in ("k", "v", "q", "alpha", "theta")]
            ms = orc.titans_forward(*a, x["eta"][b], x["m0"][b], zero)[1] if rule == "titans" else orc.delta_forward(*a, x["m0"][b])[1]
            assert_close("m", host(m)[b], ms.reshape(s + 1, -1)[-1], 1e-4)
