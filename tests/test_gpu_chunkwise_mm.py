"""GPU parity of the matrix-form (matrix-core) chunkwise Titans rule against the CPU
oracle of the frozen-M0 chunkwise rule.  Inputs k, v, q are bf16 (or float); the oracle
runs in float32 on the same (bf16-rounded) values.  Stated tolerance for bf16-input /
fp32-accumulate paths is relative 2e-2.  The bf16 forward carries every fp32 operand as a
hi + lo bf16 pair and is held to 1e-3; the bf16 backward feeds its fp32 operands to the
matrix cores as single bf16 values (fp32 accumulation) and is held to 1e-2; the float
entry points compute in fp32 throughout and are held to 1e-4 (measured: below 3e-6)."""
import numpy as np
import pytest
import torch

from nl_hecate_amd import dispatch as D
from nl_hecate_amd.ffi import lib
from oracle import pyoracle as orc
from tests.gpu_util import assert_close, dev, host, rule_inputs, zeros
from tests.test_gpu_exact_mm import kernels_run

pytestmark = pytest.mark.gpu


def bf16_round(x):
    return torch.from_numpy(x).to(torch.bfloat16).to(torch.float32).numpy()


def make(B, s, d, seed, bf16, m0_scale=0.1):
    x = rule_inputs(B, s, d, seed, m0_scale=m0_scale)
    if bf16:
        for n in ("k", "v", "q"):
            x[n] = bf16_round(x[n])
    return x


def oracle_chunkwise(x, C):
    B = x["k"].shape[0]
    fw, bw = [], []
    for b in range(B):
        a = [x[n][b] for n in ("k", "v", "q", "alpha", "theta", "eta")]
        y, mc, sc = orc.chunkwise_forward(*a, x["m0"][b], x["s0"][b], C, True)
        fw.append((y, mc, sc))
        bw.append(orc.chunkwise_backward(*a, mc, sc, x["dy"][b], C, True))
    out = dict(y=np.stack([f[0] for f in fw]), mc=np.stack([f[1] for f in fw]), sc=np.stack([f[2] for f in fw]))
    g = {n: np.stack([o[n] for o in bw]) for n in bw[0] if n not in ("d_m", "d_s")}
    g["d_m_initial"] = sum(o["d_m"] for o in bw)
    g["d_s_initial"] = sum(o["d_s"] for o in bw)
    return out, g


def gpu_forward(x, C, bf16):
    B, s, d = x["k"].shape
    nc = (s + C - 1) // C
    cv = (lambda a: dev(a).to(torch.bfloat16).contiguous()) if bf16 else dev
    k, v, q = cv(x["k"]), cv(x["v"]), cv(x["q"])
    al, th, et = dev(x["alpha"]), dev(x["theta"]), dev(x["eta"])
    mc, sc, y = zeros(B, nc + 1, d, d), zeros(B, nc + 1, d, d), zeros(B, s, d)
    name = "titans_chunkwise_forward_bf16_rocm" if bf16 else "titans_chunkwise_forward_mm_f32_rocm"
    D.call(name, k, v, q, al, th, et, dev(x["m0"]), dev(x["s0"]), mc, sc, y, s, d, B, C)
    torch.cuda.synchronize()
    return dict(k=k, v=v, q=q, al=al, th=th, et=et, mc=mc, sc=sc, y=y)


CASES = [  # B, s, C
    (2, 128, 64),
    (3, 200, 64),    # remainder chunk of 8 tokens
    (2, 96, 32),
    (2, 50, 16),     # remainder of 2
    (1, 37, 64),     # single partial chunk, odd length
    (2, 24, 1),
    (1, 1, 64),      # one token
    (5, 64, 7),      # odd chunk length, remainder of 1
    (300, 70, 64),   # more chunks (600) than compute units: the gradient kernel of bf16 tokens loops over ragged ranges, the local pass of
                     # float tokens runs two workgroups a compute unit
]


@pytest.mark.parametrize("B,s,C", CASES)
@pytest.mark.parametrize("bf16", [True, False])
def test_forward_matches_oracle(B, s, C, bf16):
    x = make(B, s, 64, seed=B * 100 + s + C, bf16=bf16)
    print(f"chunkwise_mm forward B={B} s={s} C={C} bf16={bf16}", flush=True)
    want, _ = oracle_chunkwise(x, C)
    got = gpu_forward(x, C, bf16)
    tol = 1e-3 if bf16 else 1e-4
    assert_close("y", host(got["y"]), want["y"], tol)
    assert_close("m_chunk_states", host(got["mc"]), want["mc"], tol)
    assert_close("s_chunk_states", host(got["sc"]), want["sc"], tol)


@pytest.mark.parametrize("B,s,C", CASES)
@pytest.mark.parametrize("bf16", [True, False])
def test_backward_matches_oracle(B, s, C, bf16):
    x = make(B, s, 64, seed=7 + B * 100 + s + C, bf16=bf16)
    print(f"chunkwise_mm backward B={B} s={s} C={C} bf16={bf16}", flush=True)
    _, want = oracle_chunkwise(x, C)
    f = gpu_forward(x, C, bf16)
    d = 64
    g = dict(d_k=zeros(B, s, d), d_v=zeros(B, s, d), d_q=zeros(B, s, d), d_alpha=zeros(B, s),
             d_theta=zeros(B, s), d_eta=zeros(B, s), d_m_initial=zeros(d, d), d_s_initial=zeros(d, d))
    name = "titans_chunkwise_backward_bf16_rocm" if bf16 else "titans_chunkwise_backward_mm_f32_rocm"
    D.call(name, f["k"], f["v"], f["q"], f["al"], f["th"], f["et"], f["mc"], f["sc"], dev(x["dy"]),
           g["d_k"], g["d_v"], g["d_q"], g["d_alpha"], g["d_theta"], g["d_eta"], g["d_m_initial"],
           g["d_s_initial"], s, d, B, C)
    torch.cuda.synchronize()
    tol = 1e-2 if bf16 else 1e-4
    for n in g:
        assert_close(n, host(g[n]), want[n], tol)


@pytest.mark.parametrize("C", [15, 16, 17, 32, 33, 47, 49, 63])
def test_coefficients_at_the_edges_of_their_blocks(C):
    """The coefficients come from four waves, 16 tokens each, that meet in composed maps: chunks that end one token before, at and
    behind a block's end, the last chunk of five tokens, retentions and etas of zero at the blocks' edges."""
    B, d = 2, 64
    s = 2 * C + 5
    x = make(B, s, d, seed=900 + C, bf16=False)
    for t in {t for t in (0, 15, 16, 31, C - 1) if t < C}:
        x["alpha"][:, t] = 1.0 if t % 2 else 0.0
        x["eta"][:, C + t] = 0.0
    print(f"chunkwise_mm coefficients C={C}", flush=True)
    want, want_g = oracle_chunkwise(x, C)
    f = gpu_forward(x, C, False)
    assert_close("y", host(f["y"]), want["y"], 1e-4)
    g = dict(d_k=zeros(B, s, d), d_v=zeros(B, s, d), d_q=zeros(B, s, d), d_alpha=zeros(B, s),
             d_theta=zeros(B, s), d_eta=zeros(B, s), d_m_initial=zeros(d, d), d_s_initial=zeros(d, d))
    D.call("titans_chunkwise_backward_mm_f32_rocm", f["k"], f["v"], f["q"], f["al"], f["th"], f["et"], f["mc"], f["sc"],
           dev(x["dy"]), g["d_k"], g["d_v"], g["d_q"], g["d_alpha"], g["d_theta"], g["d_eta"], g["d_m_initial"],
           g["d_s_initial"], s, d, B, C)
    torch.cuda.synchronize()
    for n in g:
        assert_close(n, host(g[n]), want_g[n], 1e-4)


@pytest.mark.parametrize("bf16", [True, False])
def test_saturated_gates(bf16):
    """alpha exactly 0 and 1 (retention 1 and 0: the memory is wiped), eta exactly 0 and 1, theta 0, at
    chunk edges and inside chunks: the coefficient tables hold exact zeros and ones there, and nothing
    in the matrix form may divide by a retention."""
    B, s, d, C = 2, 150, 64, 64
    x = make(B, s, d, seed=41, bf16=bf16)
    for t, (a, e, th) in {0: (0.0, 1.0, None), 5: (1.0, 0.0, None), 63: (1.0, 1.0, 0.0), 64: (0.0, 0.0, None),
                          100: (1.0, None, None), 128: (None, 0.0, 0.0), 149: (1.0, 1.0, None)}.items():
        if a is not None: x["alpha"][:, t] = a
        if e is not None: x["eta"][:, t] = e
        if th is not None: x["theta"][:, t] = th
    x["alpha"][1, 20:40] = 0.0   # a run of exact retention
    x["eta"][1, 70:90] = 1.0     # a run of undamped momentum
    fw, want = oracle_chunkwise(x, C)
    f = gpu_forward(x, C, bf16)
    tol = 1e-3 if bf16 else 1e-4
    assert_close("y", host(f["y"]), fw["y"], tol)
    assert_close("m_chunk_states", host(f["mc"]), fw["mc"], tol)
    assert_close("s_chunk_states", host(f["sc"]), fw["sc"], tol)
    g = dict(d_k=zeros(B, s, d), d_v=zeros(B, s, d), d_q=zeros(B, s, d), d_alpha=zeros(B, s),
             d_theta=zeros(B, s), d_eta=zeros(B, s), d_m_initial=zeros(d, d), d_s_initial=zeros(d, d))
    name = "titans_chunkwise_backward_bf16_rocm" if bf16 else "titans_chunkwise_backward_mm_f32_rocm"
    D.call(name, f["k"], f["v"], f["q"], f["al"], f["th"], f["et"], f["mc"], f["sc"], dev(x["dy"]),
           *[g[n] for n in g], s, d, B, C)
    torch.cuda.synchronize()
    tol = 1e-2 if bf16 else 1e-4
    for n in g:
        assert np.isfinite(host(g[n])).all(), n
        assert_close(n, host(g[n]), want[n], tol)


def test_launch_stream_can_be_set_and_results_are_deterministic():
    """nlh_set_stream moves every launch of an entry point (scratch clears included) to the given
    stream; the results are bit-identical to the null-stream run and to a second run."""
    import ctypes
    from nl_hecate_amd.ffi import lib
    B, s, d, C = 3, 200, 64, 64
    x = make(B, s, d, seed=17, bf16=True)

    def run():
        f = gpu_forward(x, C, True)
        g = dict(d_k=zeros(B, s, d), d_v=zeros(B, s, d), d_q=zeros(B, s, d), d_alpha=zeros(B, s),
                 d_theta=zeros(B, s), d_eta=zeros(B, s), d_m_initial=zeros(d, d), d_s_initial=zeros(d, d))
        D.call("titans_chunkwise_backward_bf16_rocm", f["k"], f["v"], f["q"], f["al"], f["th"], f["et"],
               f["mc"], f["sc"], dev(x["dy"]), *[g[n] for n in g], s, d, B, C)
        torch.cuda.synchronize()
        out = {n: host(t) for n, t in g.items()}
        out.update(y=host(f["y"]), mc=host(f["mc"]), sc=host(f["sc"]))
        return out

    a = run()
    b = run()
    side = torch.cuda.Stream()
    try:
        with torch.cuda.stream(side):
            lib.nlh_set_stream(ctypes.c_void_p(side.cuda_stream))
            c = run()
    finally:
        lib.nlh_set_stream(None)
    for n in a:
        assert np.array_equal(a[n], b[n]), f"{n}: two runs differ"
        assert np.array_equal(a[n], c[n]), f"{n}: differs on a side stream"


def test_initial_state_gradients_accumulate():
    x = make(2, 64, 64, seed=3, bf16=False)
    _, want = oracle_chunkwise(x, 32)
    f = gpu_forward(x, 32, False)
    B, s, d = 2, 64, 64
    junk = [zeros(B, s, d) for _ in range(3)] + [zeros(B, s) for _ in range(3)]
    dm, ds = torch.ones(d, d, device="cuda"), torch.ones(d, d, device="cuda")
    D.call("titans_chunkwise_backward_mm_f32_rocm", f["k"], f["v"], f["q"], f["al"], f["th"], f["et"],
           f["mc"], f["sc"], dev(x["dy"]), *junk, dm, ds, s, d, B, 32)
    torch.cuda.synchronize()
    assert_close("d_m_initial", host(dm) - 1.0, want["d_m_initial"], 1e-4)
    assert_close("d_s_initial", host(ds) - 1.0, want["d_s_initial"], 1e-4)


def test_matrix_form_agrees_with_sequential_kernels_at_benchmark_shape():
    """A second opinion beside the oracle (which checks all 128 chains of this shape in
    test_gpu_fullsize_values.py): B' = 16 chains of the config-3 shape (seq 4096, C = 64) against the
    sequential frozen-M0 kernels of the library.
    The reference-named symbols take the matrix form themselves when no clip is set, so the
    yardstick is called with an error clip that is active and never reached (1e30): that
    selects the sequential kernels and leaves every error unchanged."""
    NEVER_REACHED = 1e30
    B, s, d, C = 16, 4096, 64, 64
    x = make(B, s, d, seed=99, bf16=True, m0_scale=0.0)
    f = gpu_forward(x, C, True)
    k, v, q = (t.to(torch.float32) for t in (f["k"], f["v"], f["q"]))
    nc = s // C
    mc, sc, y = zeros(B, nc + 1, d, d), zeros(B, nc + 1, d, d), zeros(B, s, d)
    F32_MAX = float(np.finfo(np.float32).max)
    D.call("titans_chunkwise_forward_f32_cuda", k, v, q, f["al"], f["th"], f["et"], dev(x["m0"]),
           dev(x["s0"]), mc, sc, y, s, d, B, C, NEVER_REACHED, F32_MAX)
    mk = lambda: dict(d_k=zeros(B, s, d), d_v=zeros(B, s, d), d_q=zeros(B, s, d), d_alpha=zeros(B, s),
                      d_theta=zeros(B, s), d_eta=zeros(B, s), d_m_initial=zeros(d, d), d_s_initial=zeros(d, d))
    g1, g2 = mk(), mk()
    dy = dev(x["dy"])
    D.call("titans_chunkwise_backward_f32_cuda", k, v, q, f["al"], f["th"], f["et"], mc, sc, dy,
           *[g1[n] for n in g1], s, d, B, C, NEVER_REACHED, F32_MAX)
    D.call("titans_chunkwise_backward_bf16_rocm", f["k"], f["v"], f["q"], f["al"], f["th"], f["et"],
           f["mc"], f["sc"], dy, *[g2[n] for n in g2], s, d, B, C)
    torch.cuda.synchronize()
    assert_close("y", host(f["y"]), host(y), 1e-3)
    assert_close("m_chunk_states", host(f["mc"]), host(mc), 1e-3)
    for n in g1:
        assert_close(n, host(g2[n]), host(g1[n]), 1e-2)


@pytest.mark.parametrize("B,s,C", [(2, 128, 64), (3, 200, 64), (2, 50, 16)])
@pytest.mark.parametrize("bf16", [True, False])
def test_delta_matrix_form_matches_oracle(B, s, C, bf16):
    d = 64
    x = make(B, s, d, seed=31 + B * 100 + s + C, bf16=bf16)
    print(f"chunkwise_mm delta B={B} s={s} C={C} bf16={bf16}", flush=True)
    fw, bw = [], []
    for b in range(B):
        a = [x[n][b] for n in ("k", "v", "q", "alpha", "theta")] + [None]
        y, mc, _ = orc.chunkwise_forward(*a, x["m0"][b], None, C, False)
        fw.append((y, mc))
        bw.append(orc.chunkwise_backward(*a, mc, None, x["dy"][b], C, False))
    nc = (s + C - 1) // C
    cv = (lambda a: dev(a).to(torch.bfloat16).contiguous()) if bf16 else dev
    k, v, q = cv(x["k"]), cv(x["v"]), cv(x["q"])
    al, th = dev(x["alpha"]), dev(x["theta"])
    mc, y = zeros(B, nc + 1, d, d), zeros(B, s, d)
    sfx = "bf16_rocm" if bf16 else "mm_f32_rocm"
    D.call("delta_chunkwise_forward_" + sfx, k, v, q, al, th, dev(x["m0"]), mc, y, s, d, B, C)
    g = dict(d_k=zeros(B, s, d), d_v=zeros(B, s, d), d_q=zeros(B, s, d), d_alpha=zeros(B, s),
             d_theta=zeros(B, s), d_m=zeros(d, d))
    D.call("delta_chunkwise_backward_" + sfx, k, v, q, al, th, mc, dev(x["dy"]), *[g[n] for n in g], s, d, B, C)
    torch.cuda.synchronize()
    tol = 1e-3 if bf16 else 1e-4
    assert_close("y", host(y), np.stack([f[0] for f in fw]), tol)
    assert_close("m_chunk_states", host(mc), np.stack([f[1] for f in fw]), tol)
    tol = 1e-2 if bf16 else 1e-4
    for n in ("d_k", "d_v", "d_q", "d_alpha", "d_theta"):
        assert_close(n, host(g[n]), np.stack([o[n] for o in bw]), tol)
    assert_close("d_m_initial", host(g["d_m"]), sum(o["d_m"] for o in bw), tol)


@pytest.mark.parametrize("entry", ["titans_chunkwise_backward_bf16_rocm", "titans_chunkwise_backward_mm_f32_rocm",
                                   "titans_chunkwise_backward_bf16_guarded_rocm", "titans_chunkwise_backward_f32_cuda",
                                   "delta_chunkwise_backward_bf16_rocm", "delta_chunkwise_backward_f32_cuda"])
def test_gradients_of_the_initial_states_are_not_dropped(entry):
    """A null d_m_initial is refused by every entry point, with and without a d_s_initial, which is not left unwritten either; with
    a bound as well, where the sequential kernels may come to write both."""
    B, s, d, C = 2, 40, 64, 16
    titans, dt = entry.startswith("titans"), torch.bfloat16 if "bf16" in entry else torch.float32
    bounds = (0.0, 1e6) if "guarded" in entry or "cuda" in entry else ()
    kvq = [torch.zeros(B, s, d, dtype=dt, device="cuda") for _ in range(3)]
    gates = [zeros(B, s) for _ in range(3 if titans else 2)]
    states = [zeros(B, 4, d, d) for _ in range(2 if titans else 1)]
    out = [zeros(B, s, d) for _ in range(3)] + [zeros(B, s) for _ in gates]
    torch.cuda.synchronize()
    lib.nlh_set_error_mode(1)
    try:
        for first in [(None, zeros(d, d)), (None, None)] if titans else [(None,)]:
            lib.nlh_clear_error()
            D.call(entry, *kvq, *gates, *states, zeros(B, s, d), *out, *first, s, d, B, C, *bounds)
            assert b"is null" in lib.nlh_last_error()
    finally:
        lib.nlh_clear_error()
        lib.nlh_set_error_mode(0)


@pytest.mark.parametrize("rule,n,s,C", [("titans", 72, 2000, 64), ("titans", 9, 2049, 8), ("delta", 72, 2000, 32)])
def test_gate_gradients_of_more_chunks_than_waves(rule, n, s, C):
    """A wave of the gate sweeps walks over several chunks, the short last ones of chains among them; each chain's gradients are
    those of a call with too few chunks for that, bit for bit, and the sums over the chains those of the parts."""
    g = torch.Generator(device="cuda").manual_seed(n + C)
    rnd = lambda *shape: torch.randn(*shape, generator=g, device="cuda")
    mats, slots = (2, -(-s // C) + 1) if rule == "titans" else (1, -(-s // C) + 1)
    kvq = [(rnd(n, s, 64) / 8).to(torch.bfloat16) for _ in range(3)]
    gates = [torch.sigmoid(rnd(n, s)) for _ in range(mats + 1)]
    m0, d_y = rnd(n, 64, 64) * 0.1, rnd(n, s, 64)

    def both(a, b):
        cut = lambda t: t[a:b].contiguous()
        x, initial = [cut(t) for t in kvq + gates], [cut(m0)] + [zeros(b - a, 64, 64)] * (mats - 1)
        states = [zeros(b - a, slots, 64, 64) for _ in range(mats)]
        out = [zeros(b - a, s, 64) for _ in range(3)] + [zeros(b - a, s) for _ in gates]
        d0 = [zeros(64, 64) for _ in range(mats)]
        D.call(f"{rule}_chunkwise_forward_bf16_rocm", *x, *initial, *states, zeros(b - a, s, 64), s, 64, b - a, C)
        D.call(f"{rule}_chunkwise_backward_bf16_rocm", *x, *states, cut(d_y), *out, *d0, s, 64, b - a, C)
        torch.cuda.synchronize()
        return out[3:], d0

    whole, d0 = both(0, n)
    cuts = [i * n // 9 for i in range(10)]
    parts = [both(a, b) for a, b in zip(cuts, cuts[1:])]
    for i, t in enumerate(whole):
        assert torch.equal(t, torch.cat([p[0][i] for p in parts])), i
    for i, t in enumerate(d0):   # n float terms in another order
        want = sum(p[1][i].double() for p in parts)
        size = sum(p[1][i].abs().double() for p in parts)
        assert ((t.double() - want).abs() <= 2 ** -24 * 2 * n * (size + 8 * size.mean())).all(), i


def _in_parts(rule, n, s, C, step, seed):
    """Forward and backward of n chains at once and of `step` at a time: outputs of each chain, sums over the chains."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda *shape: torch.randn(*shape, generator=g, device="cuda")
    mats, slots = (2, -(-s // C) + 1) if rule == "titans" else (1, -(-s // C) + 1)
    kvq = [(rnd(n, s, 64) / 8).to(torch.bfloat16) for _ in range(3)]
    gates = [torch.sigmoid(rnd(n, s)) for _ in range(mats + 1)]
    initial, d_y = [rnd(n, 64, 64) * 0.1 for _ in range(mats)], rnd(n, s, 64)

    def both(a, b):
        cut = lambda t: t[a:b].contiguous()
        x, first = [cut(t) for t in kvq + gates], [cut(t) for t in initial]
        states, y = [zeros(b - a, slots, 64, 64) for _ in range(mats)], zeros(b - a, s, 64)
        out = [zeros(b - a, s, 64) for _ in range(3)] + [zeros(b - a, s) for _ in gates]
        d0 = [zeros(64, 64) for _ in range(mats)]
        D.call(f"{rule}_chunkwise_forward_bf16_rocm", *x, *first, *states, y, s, 64, b - a, C)
        D.call(f"{rule}_chunkwise_backward_bf16_rocm", *x, *states, cut(d_y), *out, *d0, s, 64, b - a, C)
        torch.cuda.synchronize()
        return [y, *states, *out], d0

    parts = [both(a, min(a + step, n)) for a in range(0, n, step)]
    return both(0, n), parts


# chains whose halves are more than the compute units, by one and by many; a chunk of one token at the end, chunks below a tile,
# one chunk alone
@pytest.mark.parametrize("rule", ["titans", "delta"])
@pytest.mark.parametrize("more,s,C", [(1, 193, 64), (9, 100, 64), (1, 64, 64), (72, 70, 17), (3, 33, 32), (130, 50, 64), (1, 5, 1),
                                      (132, 513, 64), (131, 100, 10)])   # the last two: the adjoint scan in halves
def test_chains_in_one_workgroup_and_in_two(rule, more, s, C):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    n = cus // 2 + more
    (whole, d0), parts = _in_parts(rule, n, s, C, 8, seed=n + s + C)
    for i, t in enumerate(whole):
        assert torch.equal(t, torch.cat([p[0][i] for p in parts])), i
    for i, t in enumerate(d0):   # n float terms in another order
        want, size = (sum(f(p[1][i].double()) for p in parts) for f in (lambda x: x, torch.abs))
        assert ((t.double() - want).abs() <= 2 ** -24 * 2 * n * (size + 8 * size.mean())).all(), i


@pytest.mark.parametrize("fires", ["nothing", "norm", "clip"])
def test_tracks_of_chains_in_one_workgroup(fires):
    """What the last chain's second half of the rows leaves behind decides alone."""
    B, s, C = torch.cuda.get_device_properties(0).multi_processor_count // 2 + 1, 130, 64
    g = torch.Generator(device="cuda").manual_seed(5)
    rnd = lambda *shape: torch.randn(*shape, generator=g, device="cuda")
    kvq = [(rnd(B, s, 64) / 8).to(torch.bfloat16) for _ in range(3)]
    gates = [torch.sigmoid(rnd(B, s) - 3) for _ in range(3)]
    m0, s0 = rnd(B, 64, 64) * 0.01, rnd(B, 64, 64) * 0.01
    if fires == "norm":
        m0[-1, 50, 3] = 1000.0
    if fires == "clip":
        kvq[1][-1, 129, 50] = 1000.0   # in the chunk of two tokens
    slots = -(-s // C) + 1
    states, y = [zeros(B, slots, 64, 64) for _ in range(2)], zeros(B, s, 64)
    ran = kernels_run(lambda: D.call("titans_chunkwise_forward_bf16_guarded_rocm", *kvq, *gates, m0, s0, *states, y, s, 64, B, C,
                                     500.0, 500.0))
    assert "cw_chain_fwd_kernel" in ran and ("rule_fwd_kernel" in ran) == (fires != "nothing"), ran
