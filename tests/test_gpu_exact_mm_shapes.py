"""The exact rules in chunk-parallel matrix form at the edges of their shapes: head size 32, intervals that a 64-token
chunk holds several of (1 = a full trajectory), ragged last chunks, momentum and none, a bound that is never reached at
head size 32, and the forward from the scan's chunk-start states, against the oracle's token loops at the fp32 bar."""
import numpy as np
import pytest
import torch

from nl_hecate_amd import dispatch as D
from nl_hecate_amd.ffi import lib
from oracle import pyoracle as orc
from tests.gpu_util import assert_close, dev, host, rule_inputs, zeros
from tests.test_gpu_chunkwise import gpu_chunkwise, oracle_chunkwise
from tests.test_gpu_exact_mm import F32_MAX, check, gpu_backward, kernels_run, oracle_pair

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def matrix_form_wherever_it_applies():
    prev = lib.nlh_exact_backward_form(1)
    yield
    lib.nlh_exact_backward_form(prev)


@pytest.mark.parametrize("B,s,d,C", [(3, 130, 32, 64), (1, 64, 32, 32), (9, 65, 32, 20), (2, 200, 32, 1), (2, 129, 64, 1),
                                     (3, 100, 64, 16), (1, 1, 32, 1), (17, 70, 32, 64)])
def test_titans_backward(B, s, d, C):
    print(B, s, d, C, flush=True)
    x = rule_inputs(B, s, d, seed=7 + s + d, m0_scale=0.02)
    cks, gs = oracle_pair(x, C)
    got = gpu_backward(x, cks, C, F32_MAX, poison=True)
    check(got, gs)
    assert "ex_grads_kernel" in got[3], got[3]


def test_titans_backward_under_a_bound_at_head_size_32():
    x = rule_inputs(3, 150, 32, seed=5, m0_scale=0.02)
    cks, gs = oracle_pair(x, 64, 1e4)
    gpu_backward(x, cks, 64, 1e4)   # a test that fired in an earlier call sends the next one to the sequential kernels
    got = gpu_backward(x, cks, 64, 1e4)
    check(got, gs)
    assert "ex_grads_kernel" in got[3] and "cw_guard_tracks_kernel" in got[3], got[3]
    top = max(np.linalg.norm(c[0].reshape(len(c[0]), -1), axis=-1).max() for c in cks)
    cks, gs = oracle_pair(x, 64, 0.5 * top)
    check(gpu_backward(x, cks, 64, 0.5 * top), gs)
    check(gpu_backward(x, cks, 64, 0.5 * top), gs)


@pytest.mark.parametrize("d", [32, 64])
def test_delta_backward_and_forward(d):
    B, s, C = 2, 140, 32
    x = rule_inputs(B, s, d, seed=31, m0_scale=0.02)
    t = {n: dev(a) for n, a in x.items()}
    nck = orc.checkpoint_count(s, C)
    mc, y = zeros(B, nck, d * d), zeros(B, s, d)
    ran = kernels_run(lambda: D.call("delta_forward_ckpt_batched_f32_rocm", t["k"], t["v"], t["q"], t["alpha"], t["theta"],
                                     t["m0"], mc, y, s, d, B, C, 0.0, F32_MAX))
    assert "ex_fwd_local_kernel" in ran, ran
    g = [zeros(B, s, d) for _ in range(3)] + [zeros(B, s) for _ in range(2)]
    dm = zeros(d, d)
    ran = kernels_run(lambda: D.call("delta_backward_ckpt_f32_rocm", t["k"], t["v"], t["q"], t["alpha"], t["theta"], mc, t["dy"],
                                     *g, dm, s, d, B, C, 0.0, F32_MAX))
    assert "ex_grads_kernel" in ran, ran
    want_dm = 0
    for b in range(B):
        a = [x[n][b] for n in ("k", "v", "q", "alpha", "theta")]
        yo, ms = orc.delta_forward(*a, x["m0"][b])
        go = orc.delta_backward(*a, ms, x["dy"][b])
        assert_close("y", host(y)[b], yo, 1e-4)
        for n, got in zip(("d_k", "d_v", "d_q", "d_alpha", "d_theta"), g):
            assert_close(n, host(got)[b], go[n], 1e-4)
        want_dm = want_dm + go["d_m"]
    assert_close("d_m_initial", host(dm), want_dm, 1e-4)


@pytest.mark.parametrize("B,s,d,C", [(2, 300, 64, 64), (1, 129, 32, 32), (3, 192, 32, 0), (2, 200, 64, 0), (9, 65, 64, 16)])
def test_titans_forward(B, s, d, C):
    """C = 0: the full trajectory, whose every slot is compared (runs of a chain meet at the chunk starts)."""
    print(B, s, d, C, flush=True)
    x = rule_inputs(B, s, d, seed=3 + s, m0_scale=0.3)
    t = {n: dev(a) for n, a in x.items()}
    n = orc.checkpoint_count(s, C) if C else s + 1
    mc, sc = (torch.full((B, n, d * d), 9.5, device="cuda") for _ in range(2))
    y = torch.full((B, s, d), 9.5, device="cuda")
    args = [t[k] for k in ("k", "v", "q", "alpha", "theta", "eta", "m0", "s0")] + [mc, sc, y, s, d, B]
    if C:
        ran = kernels_run(lambda: D.call("titans_forward_ckpt_batched_f32_rocm", *args, C, 0.0, F32_MAX))
    else:
        ran = kernels_run(lambda: D.call("titans_forward_f32_cuda", *args, s, d * d, 0.0, F32_MAX))
    assert "ex_fwd_local_kernel" in ran, ran
    for b in range(B):
        a = [x[k][b] for k in ("k", "v", "q", "alpha", "theta", "eta")]
        yo, ms, ss = orc.titans_forward(*a, x["m0"][b], x["s0"][b])
        if C:
            keep = [0] + [i + 1 for i in range(s) if (i + 1) % C == 0 or i + 1 == s]
            ms, ss = ms.reshape(s + 1, -1)[keep], ss.reshape(s + 1, -1)[keep]
        assert_close("y", host(y)[b], yo, 1e-4)
        assert_close("m", host(mc)[b], ms.reshape(n, -1), 1e-4)
        assert_close("s", host(sc)[b], ss.reshape(n, -1), 1e-4)


@pytest.mark.parametrize("has_s", [True, False])
@pytest.mark.parametrize("B,s,C,bound", [(3, 130, 64, F32_MAX), (2, 200, 20, F32_MAX), (9, 65, 16, F32_MAX), (1, 40, 1, F32_MAX),
                                         (2, 64, 64, F32_MAX), (3, 150, 32, 1e4)])
def test_frozen_rule_at_head_size_32(has_s, B, s, C, bound):
    """The frozen-M0 chunkwise rule in the same kernels; its chunks are the caller's (one chunk: the plain walk forward)."""
    print(has_s, B, s, C, bound, flush=True)
    x = rule_inputs(B, s, 32, seed=11 + s + C, m0_scale=0.05)
    (fo, go), got = oracle_chunkwise(x, C, has_s, mx=bound), []
    gpu_chunkwise(x, C, has_s, mx=bound)   # a test that fired in an earlier call sends the next one to the sequential kernels
    ran = kernels_run(lambda: got.extend(gpu_chunkwise(x, C, has_s, mx=bound)))
    assert "ex_grads_kernel" in ran and ("ex_fwd_local_kernel" in ran) == (s > C), ran
    for n in ("y", "mc") + (("sc",) if has_s else ()):
        assert_close(n, got[0][n], fo[n], 1e-4)
    for n in go:
        assert_close(n, got[1][n], go[n], 1e-4)


@pytest.mark.parametrize("rule,d", [("titans", 32), ("delta", 32), ("titans", 64)])
def test_gate_gradients_of_more_chunks_than_waves(rule, d):
    """The gate sweeps in float64 where a wave walks over several chunks (sixteen waves a compute unit are there at most), the short
    last ones of chains among them: the gate gradients of every chain are those of a call with too few chunks for that, bit for
    bit."""
    C, per_chain, titans = 64, 65, rule == "titans"
    n, s = 16 * torch.cuda.get_device_properties(0).multi_processor_count // per_chain + 2, 64 * (per_chain - 1) + 5
    print(rule, d, n, s, flush=True)
    g = torch.Generator(device="cuda").manual_seed(d + titans)
    rnd = lambda *shape: torch.randn(*shape, generator=g, device="cuda")
    k, q = (x / x.norm(dim=-1, keepdim=True) for x in (rnd(n, s, d), rnd(n, s, d)))
    gates = [torch.sigmoid(rnd(n, s)) for _ in range(3 if titans else 2)]
    x, m0, d_y = [k, rnd(n, s, d), q] + gates, rnd(n, d * d) * 0.02, rnd(n, s, d)
    slots = orc.checkpoint_count(s, C)

    def both(a, b):
        cut = lambda t: t[a:b].contiguous()
        args, states = [cut(t) for t in x], [zeros(b - a, slots, d * d) for _ in range(2 if titans else 1)]
        initial = [cut(m0)] + [zeros(b - a, d * d)] * (len(states) - 1)
        out = [zeros(b - a, s, d) for _ in range(3)] + [zeros(b - a, s) for _ in gates]
        first = [zeros(d, d) for _ in states]
        D.call(f"{rule}_forward_ckpt_batched_f32_rocm", *args, *initial, *states, zeros(b - a, s, d), s, d, b - a, C, 0.0, F32_MAX)
        ran = kernels_run(lambda: D.call(f"{rule}_backward_ckpt_f32_rocm", *args, *states, cut(d_y), *out, *first, s, d, b - a, C,
                                         0.0, F32_MAX))
        assert "cw_gates_sweep_kernel" in ran, ran
        return [out[3]] + out[5:]

    whole = both(0, n)
    cuts = [i * n // 9 for i in range(10)]
    parts = [both(a, b) for a, b in zip(cuts, cuts[1:])]
    for i, t in enumerate(whole):
        assert t.isfinite().all() and torch.equal(t, torch.cat([p[i] for p in parts])), i
