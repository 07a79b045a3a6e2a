"""The one-call decode step (decode_token_rocm) at the edges of its kernels: every head size it serves, windows that end
on and off an attention slice of 128 keys, an odd vocabulary, a persistent prefix, clamps, clip and norm bound, against
the CPU composition of the same step (oracle/serving.py)."""
import types

import numpy as np
import pytest
import torch

from nl_hecate_amd import serving as SG
from nl_hecate_amd.cms import ContextState, Pulse
from nl_hecate_amd.ffi import lib
from nl_hecate_amd.mag_layer import MemoryLevelParams
from nl_hecate_amd.memory_level import LevelConfig
from oracle import serving as SV
from tests.gpu_util import assert_close, dev, host
from tests.test_gpu_serving import gpu_params, model

pytestmark = pytest.mark.gpu
f32 = np.float32

CASES = [  # rule, active, n_persistent, heads, head size, window, prompt, tokens, vocab, level options
    ("titans", [True, True, False], 0, 2, 64, 128, 126, 4, 64, {}),
    ("delta", [True, False], 0, 3, 32, 130, 140, 3, 37, dict(m_norm_max=0.5, error_clip=0.1)),
    ("titans", [True], 3, 1, 128, 257, 300, 2, 1000, dict(alpha_floor=0.2, theta_ceil=0.03, m_norm_max=0.7)),
    ("hebbian", [False, True], 0, 2, 32, 7, 5, 4, 4, dict(m_norm_max=0.9)),
    ("dgd", [True, True, True, False], 1, 4, 64, 16, 1, 3, 130, dict(m_norm_max=1.0, error_clip=0.5)),
]


@pytest.mark.parametrize("rule,active,n_p,nh,hd,window,s,extra,v,opts", CASES)
def test_one_call_step(rule, active, n_p, nh, hd, window, s, extra, v, opts):
    print(rule, nh, hd, window, s, v, flush=True)
    d, k = nh * hd, len(active)
    p = model(d, v, k, 91 + hd)
    lcfgs = [LevelConfig(rule, nh, hd, **opts) for _ in range(k)]
    ocfg = types.SimpleNamespace(d_model=d, num_heads=nh, head_dim=hd, window_size=window, n_persistent=n_p, levels=lcfgs)
    cfg = SG.ServeConfig(d, v, nh, hd, window, s, lcfgs, n_persistent=n_p, decode_tokens=extra)
    r = np.random.default_rng(7)
    ids = r.integers(0, v, s + extra)
    mem0 = [(0.2 * r.standard_normal((nh, hd, hd))).astype(f32) for _ in range(k)]
    gp, pulse = gpu_params(p), Pulse(0, list(active))
    ctx = ContextState([dev(m.reshape(nh, hd * hd)) for m in mem0])
    _, kv = SG.gpu_prefill_forward(gp, cfg, ids, pulse, ctx)
    want, mem, kc, vc = SV.forward_all(p, ocfg, ids[:s], active, mem0)
    scale = np.abs(want).max()
    ws = SG.DecodeWorkspace(d, v)
    lib.nlh_kernel_timer_enable(1)
    for i in range(extra):
        step = SG.gpu_single_token_forward(gp, cfg, int(ids[s + i]), pulse, ctx, kv, ws)
        ref, mem, kc, vc = SV.single_token(p, ocfg, int(ids[s + i]), active, mem, kc, vc)
        assert np.abs(step - ref).max() <= 2e-2 * scale, i     # attention storage in bf16, as the other decode tests
        assert np.array_equal(host(ws.logits_gpu)[0], step)
    import ctypes
    buf = ctypes.create_string_buffer(4096)
    lib.nlh_kernel_timer_report(buf, 4096)
    lib.nlh_kernel_timer_enable(0)
    assert f"decode_logits_kernel:{extra}:".encode() in buf.value, buf.value
    for lv in range(k):
        assert_close(f"memory[{lv}]", host(ctx.memory[lv]).reshape(mem[lv].shape), mem[lv], 1e-4)


@pytest.mark.parametrize("rule,active,n_p,nh,hd,window,s,v,opts", [
    ("titans", [True, True, True], 0, 2, 64, 100, 200, 64, {}),          # final states by the chunk maps' scan
    ("titans", [True, False], 2, 3, 32, 64, 65, 33, dict(alpha_floor=0.2)),
    ("delta", [True, True], 0, 2, 32, 16, 193, 40, dict(theta_ceil=0.05)),
    ("dgd", [True], 0, 1, 128, 8, 7, 12, {}),
    ("titans", [False, False], 0, 2, 64, 8, 3, 8, {})])
def test_prefill_in_one_batch(rule, active, n_p, nh, hd, window, s, v, opts):
    """Prompts through the batched path (no per-token outputs, memories straight to their final states)."""
    print(rule, active, nh, hd, s, flush=True)
    d, k = nh * hd, len(active)
    p = model(d, v, k, 17 + s)
    lcfgs = [LevelConfig(rule, nh, hd, **opts) for _ in range(k)]
    ocfg = types.SimpleNamespace(d_model=d, num_heads=nh, head_dim=hd, window_size=window, n_persistent=n_p, levels=lcfgs)
    cfg = SG.ServeConfig(d, v, nh, hd, window, s, lcfgs, n_persistent=n_p, decode_tokens=1)
    r = np.random.default_rng(11)
    ids = r.integers(0, v, s + 1)
    mem0 = [(0.2 * r.standard_normal((nh, hd, hd))).astype(f32) for _ in range(k)]
    gp, pulse = gpu_params(p), Pulse(0, list(active))
    ctx = ContextState([dev(m.reshape(nh, hd * hd)) for m in mem0])
    prev = lib.nlh_exact_backward_form(1)   # the matrix form wherever it applies
    assert SG._prefill_in_batch(gp, cfg, ids, pulse, ContextState([m.clone() for m in ctx.memory])) is not None
    logits, kv = SG.gpu_prefill_forward(gp, cfg, ids, pulse, ctx)
    lib.nlh_exact_backward_form(prev)
    want, mem, kc, vc = SV.forward_all(p, ocfg, ids[:s], active, mem0)
    assert np.abs(logits - want[s - 1]).max() <= 2e-2 * np.abs(want).max()
    assert kv.len == s and kv.max_len == s + 1
    for got, ref in ((kv.k_cache_bf16, kc), (kv.v_cache_bf16, vc)):
        a, b = host(got.float())[:s], SV.orc.bf16_to_f32(ref)
        assert np.abs(a - b).max() <= 2 ** -7 * np.abs(b).max()
        assert not host(got.float())[s:].any()
    for lv in range(k):
        assert_close(f"memory[{lv}]", host(ctx.memory[lv]).reshape(mem[lv].shape), mem[lv], 1e-4)


@pytest.mark.parametrize("change", ["transpose", "options"])
def test_step_after_a_change_in_place(change):
    """The workspace keeps the argument block of a step: a weight transposed where it stands (same tensor, address and
    shape) or a level's option changed between two steps has to reach the second one."""
    nh, hd, v, s = 2, 32, 50, 9
    d = nh * hd
    r = np.random.default_rng(5)
    ids = r.integers(0, v, s + 2)
    mem0 = (0.2 * r.standard_normal((nh, hd * hd))).astype(f32)

    def steps(fresh):
        gp = gpu_params(model(d, v, 1, 3))
        cfg = SG.ServeConfig(d, v, nh, hd, 16, s, [LevelConfig("delta", nh, hd)], decode_tokens=2)
        ctx, pulse = ContextState([dev(mem0)]), Pulse(0, [True])
        _, kv = SG.gpu_prefill_forward(gp, cfg, ids, pulse, ctx)
        ws = SG.DecodeWorkspace(d, v)
        SG.gpu_single_token_forward(gp, cfg, int(ids[s]), pulse, ctx, kv, ws)
        if change == "transpose":
            gp.w_q.t_()
            if fresh:
                gp.w_q = gp.w_q.contiguous()
        else:
            cfg.levels[0].theta_ceil = 0.01
        if fresh:
            ws = SG.DecodeWorkspace(d, v)
        out = SG.gpu_single_token_forward(gp, cfg, int(ids[s + 1]), pulse, ctx, kv, ws)
        return out, host(ctx.memory[0])

    (a, ma), (b, mb) = steps(False), steps(True)
    assert np.abs(a - b).max() <= 2e-2 * np.abs(b).max()   # the two routes of a step round their attention to bf16
    assert_close("memory", ma, mb, 1e-5)


@pytest.mark.parametrize("kind", [np.int64, np.int32, np.uint8, lambda t: torch.tensor(t), lambda t: torch.tensor(t).cuda(), float])
def test_token_id_of_any_whole_number_type(kind):
    """The greedy loop passes np.argmax of the logits on: any whole number reaches the embedding row that an int reaches."""
    nh, hd, v, s = 2, 32, 50, 9
    d = nh * hd
    ids = np.random.default_rng(6).integers(0, v, s)
    gp = gpu_params(model(d, v, 1, 4))
    cfg = SG.ServeConfig(d, v, nh, hd, 16, s, [LevelConfig("delta", nh, hd)], decode_tokens=2)
    mem0 = np.zeros((nh, hd * hd), f32)

    def step(token):
        ctx, pulse = ContextState([dev(mem0)]), Pulse(0, [True])
        _, kv = SG.gpu_prefill_forward(gp, cfg, ids, pulse, ctx)
        return SG.gpu_single_token_forward(gp, cfg, token, pulse, ctx, kv, SG.DecodeWorkspace(d, v))

    assert np.array_equal(step(kind(v - 1)), step(v - 1))
    for bad in (v, -1):
        with pytest.raises(ValueError):
            step(np.int64(bad))


def small(rule="delta", levels=1, seed=4):
    """A prefilled model of two heads of 32 -> (params, config, pulse, context, cache, workspace)."""
    nh, hd, v, s = 2, 32, 50, 9
    d = nh * hd
    gp = gpu_params(model(d, v, levels, seed))
    cfg = SG.ServeConfig(d, v, nh, hd, 16, s, [LevelConfig(rule, nh, hd) for _ in range(levels)], decode_tokens=2)
    ctx, pulse = ContextState([dev(np.full((nh, hd * hd), 0.01, f32)) for _ in range(levels)]), Pulse(0, [True] * levels)
    _, kv = SG.gpu_prefill_forward(gp, cfg, np.random.default_rng(6).integers(0, v, s), pulse, ctx)
    return gp, cfg, pulse, ctx, kv, SG.DecodeWorkspace(d, v)


@pytest.mark.parametrize("which", ["w_q", "w_unembed", "level.w_k", "level.w_alpha", "level.b_alpha", "memory", "short cache",
                                   "float cache"])
def test_one_call_step_leaves_other_types_and_sizes_alone(which):
    """Only the two caches are bf16: any other 16-bit tensor, and a cache of floats or of fewer rows than it says, is left
    to the step by operations, which refuses it or converts."""
    gp, cfg, pulse, ctx, kv, ws = small()
    tensors = [gp.w_embed, gp.w_q, gp.w_k, gp.w_v, gp.w_o, gp.w_unembed, kv.k_cache_bf16, kv.v_cache_bf16]
    lp = gp.levels[0]
    names = dict(w_q=1, w_unembed=5) | {"level.w_k": 8, "level.w_alpha": 11, "level.b_alpha": 12, "memory": 15, "short cache": 6,
                                        "float cache": 7}
    tensors += [lp.w_k, lp.w_v, lp.w_q, lp.w_alpha, lp.b_alpha, lp.w_theta, lp.b_theta, ctx.memory[0]]
    plan = lambda: SG._decode_plan(gp, cfg, (True,), ctx, kv, ws, tensors)
    assert plan() is not None
    t = tensors[names[which]]
    tensors[names[which]] = t[:-1] if which == "short cache" else t.float() if which == "float cache" else t.to(torch.bfloat16)
    assert plan() is None


def test_prefill_with_a_padded_unembedding():
    """Columns past the vocabulary (padding to a round number) come back with the others, as from a plain product."""
    gp, cfg, pulse, _, _, _ = small()
    v = cfg.vocab_size
    ids = np.random.default_rng(8).integers(0, v, cfg.seq_len)
    memory = lambda: ContextState([dev(np.full((cfg.num_heads, cfg.head_dim ** 2), 0.01, f32))])
    want, _ = SG.gpu_prefill_forward(gp, cfg, ids, pulse, memory())
    gp.w_unembed = torch.cat([gp.w_unembed, torch.full((cfg.d_model, 6), 3.0, device="cuda")], 1).contiguous()
    assert SG._prefill_in_batch(gp, cfg, ids, pulse, memory()) is None
    got, _ = SG.gpu_prefill_forward(gp, cfg, ids, pulse, memory())
    assert got.shape == (v + 6,) and np.abs(got[:v] - want).max() <= 2e-2 * np.abs(want).max()


@pytest.mark.parametrize("gate", ["b_alpha", "w_theta"])
@pytest.mark.parametrize("opts,finite", [({}, False), (dict(alpha_ceil=0.9, theta_ceil=2.0), True),
                                         (dict(alpha_floor=0.8, alpha_ceil=0.3, theta_floor=0.5, theta_ceil=0.2), True)])
def test_nan_of_a_gate_parameter(gate, opts, finite):
    """Without bounds a NaN of a gate's parameters reaches the logits and the memory, of a token and of a prompt; bounds
    that are set replace it (by the ceiling, or the floor where that is higher), as the clamp of the level step does."""
    gp, cfg, pulse, ctx, kv, ws = small()
    clean = host(ctx.memory[0])
    for k, x in opts.items():
        setattr(cfg.levels[0], k, x)
    getattr(gp.levels[0], gate)[0] = float("nan")
    step = SG.gpu_single_token_forward(gp, cfg, 3, pulse, ctx, kv, ws)
    assert np.isfinite(step).all() == finite and np.isfinite(host(ctx.memory[0])).all() == finite
    ids = np.arange(cfg.seq_len)
    ctx = ContextState([dev(clean)])
    assert SG._prefill_in_batch(gp, cfg, ids, pulse, ContextState([dev(clean)])) is not None
    logits, _ = SG.gpu_prefill_forward(gp, cfg, ids, pulse, ctx)
    assert np.isfinite(logits).all() == finite and np.isfinite(host(ctx.memory[0])).all() == finite
    if gate == "b_alpha" and finite:   # the same as a bias that drives the gate to that bound
        gp.levels[0].b_alpha[0] = 1e30
        want = ContextState([dev(clean)])
        SG.gpu_prefill_forward(gp, cfg, ids, pulse, want)
        assert np.array_equal(host(ctx.memory[0]), host(want.memory[0]))


@pytest.mark.parametrize("name", ["logits_gpu", "embedded", "gated_out", "attn_out_bf16", "logits_host"])
def test_step_after_a_workspace_buffer_was_replaced(name):
    """The kept argument block holds the workspace's addresses: a buffer put in another's place is the one written."""
    gp, cfg, pulse, ctx, kv, ws = small()
    first = ctx.memory[0].clone()
    want = SG.gpu_single_token_forward(gp, cfg, 3, pulse, ctx, kv, ws)
    old, filled = getattr(ws, name), host(getattr(ws, name).clone().float())
    setattr(ws, name, torch.zeros_like(old, pin_memory=name == "logits_host"))
    old.fill_(7.0)
    ctx.memory[0].copy_(first)
    kv.len -= 1
    assert np.array_equal(SG.gpu_single_token_forward(gp, cfg, 3, pulse, ctx, kv, ws), want)
    assert np.array_equal(host(getattr(ws, name).float()), filled) and (host(old.float()) == 7.0).all()


def test_windows_past_what_one_call_merges():
    """head-slices of 128 keys beyond the merge's LDS go step by operations; a window without an end costs no memory."""
    nh, hd, v, s = 128, 32, 8, 12400    # 97 slices of 128 heads and a width of 4096: 128 floats past 64 KB
    d = nh * hd
    cfg = SG.ServeConfig(d, v, nh, hd, 1 << 30, s, [LevelConfig("hebbian", nh, hd)])
    assert not SG._keys_fit(cfg, s - 1) and SG._keys_fit(cfg, 96 * 128 - 1)
    g = torch.Generator(device="cuda").manual_seed(1)
    r = lambda *sh: torch.randn(*sh, generator=g, device="cuda") * 0.02
    gp = SG.GpuMAGParams(r(v, d), r(d, d), r(d, d), r(d, d), r(d, d), r(d, v),
                         [MemoryLevelParams(r(d, d), r(d, d), r(d, d), r(2 * d), r(1), r(2 * d), r(1), r(2 * d), r(1))])
    kv = SG.GpuKVCache(s + 4, d, 1)
    kv.k_cache_bf16.copy_(r(s + 4, d) * 50)
    kv.v_cache_bf16.copy_(r(s + 4, d) * 50)
    out = []
    for window, start in ((16000, s), (1 << 30, 96 * 128 - 2)):
        cfg.window_size, kv.len = window, start
        ws = SG.DecodeWorkspace(d, v)
        ctx = ContextState([torch.zeros(nh, hd * hd, device="cuda")])
        out.append(SG.gpu_single_token_forward(gp, cfg, 1, Pulse(0, [True]), ctx, kv, ws))
        assert bool(ws.plans) == (start < s) and ws.work.numel() < 1 << 20
        q, keys = (host(x.float()).astype(np.float64) for x in (ws.q_bf16, kv.k_cache_bf16[:start + 1]))
        w = np.einsum("hc,thc->ht", q.reshape(nh, hd), keys.reshape(-1, nh, hd)) / np.sqrt(hd)
        w = np.exp(w - w.max(1, keepdims=True))
        w /= w.sum(1, keepdims=True)
        want = np.einsum("ht,thc->hc", w, host(kv.v_cache_bf16[:start + 1].float()).reshape(-1, nh, hd))
        assert np.abs(host(ws.attn_out).reshape(nh, hd) - want).max() <= 2e-2 * np.abs(want).max()
    assert np.isfinite(out).all()


@pytest.mark.parametrize("how", ["deepcopy", "pickle"])
def test_a_used_workspace_can_be_copied_and_saved(how):
    import copy
    import pickle
    gp, cfg, pulse, ctx, kv, ws = small()
    first = ctx.memory[0].clone()
    want = SG.gpu_single_token_forward(gp, cfg, 3, pulse, ctx, kv, ws)
    other = copy.deepcopy(ws) if how == "deepcopy" else pickle.loads(pickle.dumps(ws))
    assert np.array_equal(host(other.logits_gpu)[0], want) and np.array_equal(other.logits_host.numpy(), want)
    ws.logits_gpu.zero_()
    ctx.memory[0].copy_(first)
    kv.len -= 1
    assert np.array_equal(SG.gpu_single_token_forward(gp, cfg, 3, pulse, ctx, kv, other), want)
    assert not host(ws.logits_gpu).any() and np.array_equal(host(other.logits_gpu)[0], want)
    assert list(other.plans.values())[0][1] is not None
    old = object.__new__(SG.DecodeWorkspace)
    old.__setstate__({n: t for n, t in ws.__getstate__().items() if n != "logits_host"})
    kv.len -= 1
    ctx.memory[0].copy_(first)
    assert np.array_equal(SG.gpu_single_token_forward(gp, cfg, 3, pulse, ctx, kv, old), want)


def test_non_finite_cache_entries(monkeypatch):
    """NaN and infinities among the cached keys and values end up where the step by operations has them."""
    gp, cfg, pulse, ctx, kv, ws = small()
    first = ctx.memory[0].clone()
    k0, v0 = kv.k_cache_bf16.clone(), kv.v_cache_bf16.clone()
    in_one = SG._decode_in_one_call
    for place in ("k nan", "k inf", "k -inf", "all k -inf", "v nan", "v inf"):
        kv.k_cache_bf16.copy_(k0)
        kv.v_cache_bf16.copy_(v0)
        cache = kv.k_cache_bf16 if "k" in place else kv.v_cache_bf16
        cache[slice(None) if "all" in place else slice(4, 5), 3 if "k" in place else 40] = float(place.split()[-1])
        out = []
        for one in (True, False):
            monkeypatch.setattr(SG, "_decode_in_one_call", in_one if one else lambda *a: None)
            ctx.memory[0].copy_(first)
            kv.len = cfg.seq_len
            SG.gpu_single_token_forward(gp, cfg, 3, pulse, ctx, kv, ws)
            out.append(host(ws.attn_out)[0].copy())
        a, b = out
        assert np.array_equal(np.isfinite(a), np.isfinite(b)), place
        ok = np.isfinite(b)
        assert np.abs(a[ok] - b[ok]).max(initial=0) <= 2e-2 * np.abs(b[ok]).max(initial=1), place


@pytest.mark.parametrize("nh,hd,levels,keys", [
    (2, 32, 5, 9 * 128 - 3),     # more levels and slices than the first batch of loads holds
    (16, 32, 1, 17 * 128 + 1),   # more statistics than threads
    (1, 32, 4, 33 * 128),        # more statistics than columns
    (10, 64, 8, 100)])           # more columns than two a thread
def test_output_merge_at_its_edges(nh, hd, levels, keys):
    d, v = nh * hd, 20
    g = torch.Generator(device="cuda").manual_seed(keys)
    r = lambda *sh: torch.randn(*sh, generator=g, device="cuda") * 0.1
    lp = [MemoryLevelParams(r(d, d), r(d, d), r(d, d), r(2 * d), r(1), r(2 * d), r(1), r(2 * d), r(1)) for _ in range(levels)]
    gp = SG.GpuMAGParams(r(v, d), r(d, d), r(d, d), r(d, d), r(d, d), r(d, v), lp)
    cfg = SG.ServeConfig(d, v, nh, hd, keys, keys - 1, [LevelConfig("delta", nh, hd) for _ in range(levels)], decode_tokens=2)
    kv, ws = SG.GpuKVCache(keys + 1, d, 1), SG.DecodeWorkspace(d, v)
    kv.k_cache_bf16.copy_(r(keys + 1, d) * 30)
    kv.v_cache_bf16.copy_(r(keys + 1, d) * 10)
    kv.len = keys - 1
    ctx = ContextState([r(nh, hd * hd) for _ in range(levels)])
    out = SG.gpu_single_token_forward(gp, cfg, 3, Pulse(0, [False] * levels), ctx, kv, ws)
    assert list(ws.plans.values())[0][1] is not None
    f64 = lambda t: host(t.float()).astype(np.float64)
    q, kc, vc = (f64(t).reshape(-1, nh, hd) for t in (ws.q_bf16, kv.k_cache_bf16[:keys], kv.v_cache_bf16[:keys]))
    w = np.einsum("hc,thc->ht", q[0], kc) / np.sqrt(hd)
    w = np.exp(w - w.max(1, keepdims=True))
    attn = np.einsum("ht,thc->hc", w / w.sum(1, keepdims=True), vc).reshape(-1)
    got = f64(ws.attn_out)[0]
    assert np.abs(got - attn).max() <= 2 ** -8 * np.abs(attn).max()   # rounded to bf16 once
    x = f64(gp.w_embed)[3]
    y = sum(np.einsum("hij,hj->hi", f64(m).reshape(nh, hd, hd), (f64(p.w_q) @ x).reshape(nh, hd))
            for m, p in zip(ctx.memory, lp)).reshape(-1) * (levels ** -0.5 if levels > 2 else 1.0)
    scale = sum(np.abs(f64(m)).max() for m in ctx.memory) * np.abs(x).max() * d * hd * 0.4
    assert np.abs(f64(ws.y_combined)[0] - y).max() <= 2e-7 * scale   # float sums of d and of hd products
    gated = got / (1 + np.exp(-f64(ws.y_combined)[0]))
    assert_close("gated", f64(ws.gated_out)[0], gated, 1e-6)
    assert_close("logits", out, (f64(gp.w_o) @ gated) @ f64(gp.w_unembed), 1e-5)
