"""Groups of levels as one batch (csrc/level_group.hip, csrc/gemm_f32.hip): the grouped products at the edges of their
tiles and splits against float64, the multi-tensor update, the register-held cross-entropy rows, and a grouped training
step against the same step level by level (whose parity with the oracle has its own tests)."""
import ctypes

import numpy as np
import pytest
import torch

from nl_hecate_amd import cms_model as GM
from nl_hecate_amd import dispatch as D
from nl_hecate_amd import memory_level as ML
from nl_hecate_amd.ffi import lib
from tests.gpu_util import dev, host
from tests.test_gpu_cms_model import gpu_model, setup
from nl_hecate_amd.cms import ContextState, Pulse

pytestmark = pytest.mark.gpu
f32 = np.float32


@pytest.mark.parametrize("op,count,m,n,k", [(0, 1, 1, 4, 4), (0, 3, 65, 36, 100), (0, 2, 300, 260, 64), (0, 17, 129, 64, 32),
                                            (0, 1, 70, 64, 8000), (1, 1, 5, 4, 4), (1, 7, 130, 128, 96), (1, 15, 512, 256, 256),
                                            (2, 4, 64, 132, 777), (2, 1, 4, 4, 1), (2, 33, 32, 64, 50)])
def test_grouped_products(op, count, m, n, k):
    print(op, count, m, n, k, flush=True)
    r = np.random.default_rng(m + n + k)
    shp_a, shp_b = {0: ((m, k), (n, k)), 1: ((m, k), (k, n)), 2: ((k, m), (k, n))}[op]
    A = [r.standard_normal(shp_a).astype(f32) for _ in range(count)]
    B = [r.standard_normal(shp_b).astype(f32) for _ in range(count)]
    a, b = [dev(x) for x in A], [dev(x) for x in B]
    c = [torch.full((m, n), 7.5, device="cuda") for _ in range(1 if op == 1 else count)]
    ML.linear_group(op, a, b, c, m, n, k)
    want = {0: lambda: [x.astype(np.float64) @ y.T for x, y in zip(A, B)],
            1: lambda: [sum(x.astype(np.float64) @ y for x, y in zip(A, B))],
            2: lambda: [x.T.astype(np.float64) @ y for x, y in zip(A, B)]}[op]()
    terms = k * (count if op == 1 else 1)
    for got, w in zip(c, want):
        # fp32 sums of `terms` products of unit normals: rounding grows like sqrt(terms) ulps of sums of size sqrt(terms)
        assert np.abs(host(got) - w).max() <= 8 * 2 ** -24 * terms + 1e-6
    if op == 0:
        half = [torch.zeros(m, n, dtype=torch.bfloat16, device="cuda") for _ in range(count)]
        ML.linear_group(0, a, b, half, m, n, k, (1 << count) - 1)
        for h, got in zip(half, c):
            assert (h.float() - got).abs().max().item() <= 2 ** -7 * got.abs().max().item()


@pytest.mark.parametrize("op,m,n,k", [(0, 1, 1, 1), (0, 257, 129, 31), (0, 300, 130, 33), (0, 512, 510, 4097), (0, 2100, 2060, 64),
                                      (1, 3, 2, 5), (1, 255, 127, 65), (1, 513, 8001, 96), (1, 130, 70, 2000), (2, 1, 3, 7),
                                      (2, 129, 1003, 50), (2, 512, 8193, 97), (2, 65, 65, 1)])
def test_single_products_of_any_size(op, m, n, k):
    print(op, m, n, k, flush=True)
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    shp_a, shp_b = {0: ((m, k), (n, k)), 1: ((m, k), (k, n)), 2: ((k, m), (k, n))}[op]
    a, b = [torch.randn(*s, generator=g, device="cuda") for s in (shp_a, shp_b)]
    c = torch.full((m * n + 4,), 7.5, device="cuda")
    ML.product(op, a, b, c, m, n, k)
    assert (c[m * n:] == 7.5).all()
    fit = {0: lambda a, b: a @ b.t(), 1: lambda a, b: a @ b, 2: lambda a, b: a.t() @ b}[op]
    want, got = fit(a.double(), b.double()), c[:m * n].view(m, n).double()
    # every product of two floats is kept to 2^-24 of it, every sum of 32 rounds; fp32 products added one by one: as above
    assert (got - want).abs().max().item() <= 8 * 2 ** -24 * k + 1e-6
    if k >= 64:   # no further from float64 than sums term by term
        assert (got - want).norm().item() <= (fit(a, b).double() - want).norm().item()
    # magnitudes: the pieces of a float follow it down to the last of a bf16's range, 2^-133
    for scale_a, scale_b in ((2. ** -90, 2. ** 80), (2. ** 100, 2. ** -60), (2. ** -112, 1.)):
        ML.product(op, a * scale_a, b * scale_b, c, m, n, k)
        assert (c[:m * n].view(m, n).double() / (scale_a * scale_b) - want).abs().max().item() <= 8 * 2 ** -24 * k + 1e-6


@pytest.mark.parametrize("op", [0, 1, 2])
@pytest.mark.parametrize("m,n,k", [(600, 1300, 64), (72, 67, 35)])
def test_single_products_keep_non_finite_values_in_their_place(op, m, n, k):
    g = torch.Generator(device="cuda").manual_seed(5)
    shp_a, shp_b = {0: ((m, k), (n, k)), 1: ((m, k), (k, n)), 2: ((k, m), (k, n))}[op]
    a, b = [torch.randn(*s, generator=g, device="cuda") for s in (shp_a, shp_b)]
    a[3, 5], a[-1, 1], b[2, 7], b[-1, -1] = float("nan"), float("inf"), -float("inf"), 3.4e38
    c = torch.zeros(m, n, device="cuda")
    ML.product(op, a, b, c, m, n, k)
    x, y = {0: (a, b.t()), 1: (a, b), 2: (a.t(), b)}[op]
    want = sum(x[:, i, None].double() * y[None, i].double() for i in range(k))
    want = torch.where(want.abs() > 3.5e38, want.sign() * float("inf"), want)
    near = (want.abs() > 3.3e38) & want.isfinite()   # a sum on either side of the largest float
    assert torch.equal(c.isnan() | near, want.isnan() | near) and torch.equal(c.isinf() | near, want.isinf() | near)
    ok = want.isfinite() & ~near
    assert ((c.double() - want)[ok].abs() <= 8 * 2 ** -24 * k * want[ok].abs().clamp(min=1)).all()


@pytest.mark.parametrize("op", [0, 1, 2])
@pytest.mark.parametrize("m,n,k", [(600, 1300, 128), (130, 70, 2000)])
def test_single_products_of_the_smallest_floats(op, m, n, k):
    """Operands whose three pieces do not hold all of their bits any more, alone and as one row among others; zeros stay."""
    g = torch.Generator(device="cuda").manual_seed(6)
    shp_a, shp_b = {0: ((m, k), (n, k)), 1: ((m, k), (k, n)), 2: ((k, m), (k, n))}[op]
    a, b = [torch.randn(*s, generator=g, device="cuda") for s in (shp_a, shp_b)]
    fit = {0: lambda a, b: a @ b.t(), 1: lambda a, b: a @ b, 2: lambda a, b: a.t() @ b}[op]
    c = torch.zeros(m, n, device="cuda")
    for scale, scale_b, row in ((2. ** -113, 1., None), (2. ** -120, 1., 5), (2. ** -122, 2. ** 20, None), (2. ** -125, 2. ** 5, m - 1)):
        x, y = a.clone(), b * scale_b
        rows = x.t() if op == 2 else x
        rows[...] = rows * scale if row is None else rows.index_copy(0, torch.tensor([row], device="cuda"), rows[row:row + 1] * scale)
        rows[7] = 0
        ML.product(op, x, y, c, m, n, k)
        want, by_terms = fit(x.double(), y.double()), fit(x, y).double()
        at = slice(None) if row is None else slice(row, row + 1)
        # sums term by term like the library's, in another order: as many roundings of sums of the same size, within twice
        assert (c.double() - want)[at].norm().item() <= 2 * (by_terms - want)[at].norm().item(), (scale, scale_b, row)
        assert (c[7] == 0).all()


@pytest.mark.parametrize("count,m,n,k", [(7, 1000, 1024, 1024), (6, 2000, 512, 512), (12, 512, 512, 512)])
def test_sum_over_products_rounds_like_products_added_up(count, m, n, k):
    g = torch.Generator(device="cuda").manual_seed(1)
    a, b = [[torch.randn(*s, generator=g, device="cuda") for _ in range(count)] for s in ((m, k), (k, n))]
    c, one = torch.zeros(m, n, device="cuda"), a[0] @ b[0]
    ML.linear_group(1, a, b, [c], m, n, k)
    for x, y in zip(a[1:], b[1:]):
        one.addmm_(x, y)
    want = sum(x.double() @ y.double() for x, y in zip(a, b))
    err = lambda t: ((t.double() - want).norm() / want.norm()).item()
    # each product rounds like one of the library's, and the sums over products add to that on both sides
    assert err(c) <= 1.05 * err(one)


def test_saxpy_multi():
    r = np.random.default_rng(3)
    sizes = [1, 3, 4096, 4097, 5, 100000, 64] * 10
    x, y = [[r.standard_normal(n).astype(f32) for n in sizes] for _ in range(2)]
    xd, yd = [dev(t) for t in x], [dev(t) for t in y]
    shifted = torch.zeros(8, device="cuda")   # an operand that is not at a 16-byte boundary
    xd.append(dev(np.arange(5, dtype=f32)))
    yd.append(shifted[1:6])
    n = [t.numel() for t in xd]
    lib.saxpy_multi_rocm(-0.25, ML._ptrs(xd), ML._ptrs(yd), (ctypes.c_int * len(n))(*n), len(n))
    for a, b, g in zip(x, y, yd):
        assert np.array_equal(host(g), (b + f32(-0.25) * a)) or np.abs(host(g) - (b - 0.25 * a)).max() <= 2 ** -23 * np.abs(b).max() * 2
    assert np.array_equal(host(shifted), np.array([0, 0, -0.25, -0.5, -0.75, -1.0, 0, 0], f32))


def test_saxpy_multi_of_shared_tensors():
    """A tensor that two pairs update takes both updates, and one that a later pair reads is read updated, as pair by pair."""
    r = np.random.default_rng(4)
    y, x = r.standard_normal(9000).astype(f32), [r.standard_normal(9000).astype(f32) for _ in range(3)]
    for _ in range(5):
        yd, xd = dev(y), [dev(t) for t in x]
        ys, xs, n = [yd, yd, yd[4000:], xd[1]], [xd[0], xd[1], xd[2], yd], [9000, 9000, 5000, 9000]
        lib.saxpy_multi_rocm(0.5, ML._ptrs(xs), ML._ptrs(ys), (ctypes.c_int * 4)(*n), 4)
        want = (y + f32(0.5) * x[0]) + f32(0.5) * x[1]
        want[4000:] += f32(0.5) * x[2][:5000]
        assert np.abs(host(yd) - want).max() <= 2e-6
        assert np.abs(host(xd[1]) - (x[1] + f32(0.5) * want)).max() <= 2e-6


@pytest.mark.parametrize("s,v", [(5, 1024), (3, 8192), (4, 8196), (2, 32768), (3, 16388), (2, 32772)])
def test_cross_entropy_rows(s, v):
    r = np.random.default_rng(v)
    x = (4 * r.standard_normal((s, v))).astype(f32)
    t = r.integers(0, v, s).astype(np.int32)
    t[0] = v - 1
    if s > 2:
        t[1] = -1
    loss, g = torch.zeros(1, device="cuda"), torch.full((s, v), 3.0, device="cuda")
    D.call("cross_entropy_forward_cuda", dev(x), dev(t), loss, s, v)
    D.call("cross_entropy_backward_cuda", dev(x), dev(t), g, s, v, 0.5)
    p = np.exp(x.astype(np.float64) - x.max(1, keepdims=True))
    p /= p.sum(1, keepdims=True)
    ok = t >= 0
    want = -np.log(p[np.arange(s), t])[ok].sum()
    assert abs(loss.item() - want) <= 1e-5 * want
    p[np.arange(s), t] -= 1
    assert np.abs(host(g) - 0.5 * p * ok[:, None]).max() <= 1e-6


@pytest.mark.parametrize("rule,k,nh,hd,s,bs,kw", [
    ("titans", 3, 2, 32, 70, 2, {}),
    ("delta", 2, 4, 8, 33, 1, dict(alpha_floor=0.3, theta_ceil=0.04, m_norm_max=0.8)),
    ("titans", 2, 3, 4, 40, 1, dict(checkpoint_interval=8, alpha_ceil=0.4)),
    ("dgd", 2, 2, 16, 50, 1, dict(error_clip=0.2)),
    ("titans", 2, 10, 64, 130, 1, dict(proxy=True, chunk_size=64, m_norm_max=50.0))])
def test_grouped_step_against_level_by_level(rule, k, nh, hd, s, bs, kw, monkeypatch):
    print(rule, k, nh, hd, s, bs, flush=True)
    cfg, _, p, mem = setup(rule, k, nh, hd, 60, s, 16, bs=bs, **kw)
    ids = [int(t) for t in np.random.default_rng(1).integers(0, 60, bs * s)]
    out = []
    for grouped in (True, False):
        if not grouped:
            for mod in (GM, ML):
                monkeypatch.setattr(mod, "group_key", lambda *a: None)
        gp, _ = gpu_model(p)
        ctx = ContextState([dev(m.reshape(m.shape[0], hd * hd)) for m in mem])
        loss, cache = GM.gpu_cms_forward(gp, cfg, ids, ids[1:] + ids[:1], Pulse(0, [True] * k), ctx)
        assert (cache["memory_caches"][0].group is not None) == grouped
        g = GM.gpu_cms_backward(gp, cfg, cache)
        GM.gpu_weight_update(gp, g, 0.1)
        vals = [torch.tensor([loss]), g.d_w_embed, g.d_w_q, g.d_w_k, g.d_w_v, g.d_w_o, g.d_w_unembed, gp.w_q, gp.w_embed, *ctx.memory]
        for lg, lp, mc in zip(g.levels, gp.levels, cache["memory_caches"]):
            vals += [lg.d_w_k_mem, lg.d_w_v_mem, lg.d_w_q_mem, lg.d_w_alpha, lg.d_b_alpha, lg.d_w_theta, lg.d_b_theta, lg.d_w_eta,
                     lg.d_b_eta, lp.w_alpha, lp.w_k, mc.k_mem, mc.q_mem, mc.alpha, mc.theta, mc.m_states]
        out.append([host(x) for x in vals])
    for i, (a, b) in enumerate(zip(*out)):
        # the attention's q, k, v may round to neighbouring bf16 where the products' sums differ in their last bits
        assert np.abs(a - b).max() <= 2e-3 * max(np.abs(b).max(), 1e-6), i


@pytest.mark.parametrize("gate", ["b_alpha", "b_theta", "w_eta"])
def test_nan_of_a_gate_parameter_reaches_the_loss(gate):
    cfg, _, p, mem = setup("titans", 2, 2, 32, 60, 40, 16)
    ids = [int(t) for t in np.random.default_rng(1).integers(0, 60, 40)]
    gp, _ = gpu_model(p)
    getattr(gp.levels[1], gate)[0] = float("nan")
    ctx = ContextState([dev(m.reshape(m.shape[0], -1)) for m in mem])
    loss, cache = GM.gpu_cms_forward(gp, cfg, ids, ids, Pulse(0, [True] * 2), ctx)
    assert cache["memory_caches"][1].group is not None
    assert np.isnan(loss) and np.isnan(host(ctx.memory[1])).any()
    g = GM.gpu_cms_backward(gp, cfg, cache)
    assert np.isnan(host(g.levels[1].d_w_alpha)).any()


def test_cross_entropy_rows_of_non_finite_logits():
    """NaN, both infinities and the type's lowest value among the logits: as the kernel of any vocabulary size."""
    v, n = 1024, 6
    x = (3 * np.random.default_rng(2).standard_normal((n, v))).astype(f32)
    x[0, 5], x[1, 7], x[2, 9] = np.nan, np.inf, -np.inf
    x[3, :], x[4, :-1] = -np.inf, np.finfo(f32).min
    out = []
    for w in (v, v + 1):     # one more column, which weighs nothing: the general kernel
        xs = np.full((n, w), -np.inf, f32)
        xs[:, :v] = x
        row = []
        for i in range(n):
            loss, g = torch.zeros(1, device="cuda"), torch.zeros(1, w, device="cuda")
            t = dev(np.array([11], np.int32))
            D.call("cross_entropy_forward_cuda", dev(xs[i:i + 1]), t, loss, 1, w)
            D.call("cross_entropy_backward_cuda", dev(xs[i:i + 1]), t, g, 1, w, 0.5)
            row.append((host(loss), host(g)[:, :v]))
        out.append(row)
    for i, (a, b) in enumerate(zip(*out)):
        for p, q in zip(a, b):
            assert np.array_equal(np.isnan(p), np.isnan(q)), i
            assert np.allclose(p, q, rtol=1e-5, atol=1e-6, equal_nan=True), i


@pytest.mark.parametrize("op", [0, 1, 2])
def test_grouped_products_keep_non_finite_values_in_their_place(op):
    m, n, k = 72, 68, 36
    r = np.random.default_rng(9)
    shp_a, shp_b = {0: ((m, k), (n, k)), 1: ((m, k), (k, n)), 2: ((k, m), (k, n))}[op]
    A, B = r.standard_normal(shp_a).astype(f32), r.standard_normal(shp_b).astype(f32)
    A[3, 5], A[6, 1], B[2, 7] = np.nan, np.inf, -np.inf
    c = torch.zeros(m, n, device="cuda")
    ML.linear_group(op, [dev(A)], [dev(B)], [c], m, n, k)
    a, b = {0: (A, B.T), 1: (A, B), 2: (A.T, B)}[op]
    with np.errstate(invalid="ignore"):
        want = (a.astype(np.float64)[:, :, None] * b.astype(np.float64)[None]).sum(1)
    assert np.array_equal(np.isnan(host(c)), np.isnan(want)) and np.array_equal(np.isinf(host(c)), np.isinf(want))


def test_levels_that_share_a_memory_take_it_in_turn():
    cfg, _, p, mem = setup("delta", 2, 2, 32, 60, 20, 16)
    ids = [int(t) for t in np.random.default_rng(1).integers(0, 60, 20)]
    gp, _ = gpu_model(p)
    one = dev(mem[0].reshape(mem[0].shape[0], -1))
    first = one.clone()
    loss, cache = GM.gpu_cms_forward(gp, cfg, ids, ids, Pulse(0, [True] * 2), ContextState([one, one]))
    # the second level starts from what the first one left
    y0, c0 = ML.gpu_memory_forward(gp.levels[0], cfg.levels[0], cache["embedded"], first, 20, 64, 1)
    y1, c1 = ML.gpu_memory_forward(gp.levels[1], cfg.levels[1], cache["embedded"], first, 20, 64, 1)
    for got, want in ((cache["y_per_level"][0], y0), (cache["y_per_level"][1], y1), (one, first)):
        assert np.array_equal(host(got), host(want))
