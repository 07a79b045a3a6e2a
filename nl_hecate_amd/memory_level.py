"""Host mirror of the reference's per-level memory step on device buffers:
gpu_memory_forward (core/src/gpu_forward.rs:1197-1705), gpu_memory_backward
(core/src/gpu_backward.rs:459-1200), accumulate_projection_grads (:2047-2117) and the
GpuMemoryCache variants of the matrix memories (gpu_forward.rs:129-312):

    Delta, Titans, Hebbian, DGD                  full trajectory  [bs*nh, s+1, hd*hd]
    DeltaCkpt, TitansCkpt, HebbianCkpt, DGDCkpt  checkpoints      [bs*nh, n_ckpt, hd*hd]
    DeltaChunkwise, TitansChunkwise              chunk states     [bs*nh, n_chunks+1, hd*hd]
    TitansMlp                                    packed MLP state [bs*nh, s+1, 2*hd*dh + dh + hd] per head
    Mlp (MONETA, YAAD)                           W1 / W2 trajectories [s+1, dh*d], [s+1, d*dh], batch 1
    SwiGlu                                       the stateless MLP's four activation buffers

Same order of operations and the same cached tensors as the reference: projections of the input,
L2 normalisation of k and q, gate projections with their clamps, per-head layout, the rule, the final
memory carried into `context_m` under its Frobenius clamp; backward: the rule's backward per head, gate
gradients summed over heads and masked where a gate sat on a clamp bound, back to token layout,
normalisation backward, projection and gate weight gradients, d_embedded.  Tensors are float32 CUDA
tensors (torch stands in for GpuBuf); every step is a call into libnl_hecate_rocm.so or, for the levels that do
not run as a group, a torch matmul for the projections (cublas_matmul_*_dd in the reference) — nothing is computed
on the host.  Delta, Titans and DGD levels with equal options run as one batch (forward_group, backward_group).

Where the reference loops single-chain kernels over heads and refuses batch_size > 1 (checkpointed
variants, gpu_forward.rs:1608-1703), the batched entry points of the library take every chain at once
and any batch size.
"""
import ctypes
from dataclasses import dataclass, field
from typing import Optional

import numpy as np
import torch

from . import dispatch as D
from .ffi import lib
from .mag_layer import MemoryLevelParams

F32_MAX = 3.4028234663852886e38
RULES = ("delta", "titans", "hebbian", "dgd", "moneta", "yaad", "swiglu")
ACTIVATIONS = {"gelu": 0, "silu": 1, "relu": 2}   # MemoryActivation -> the kernels' activation id


@dataclass
class LevelConfig:
    """What gpu_memory_forward / gpu_memory_backward read from MAGConfig for one level."""
    memory_rule: str                            # MemoryRuleKind: "delta", "titans", "hebbian", "dgd"
    num_heads: int                              # cfg.swa.num_heads
    head_dim: int                               # cfg.swa.head_dim
    checkpoint_interval: Optional[int] = None   # effective_checkpoint_interval(level)
    proxy: bool = False                         # tape_strategy_for_level(level) == Proxy: frozen-M0 chunkwise
    chunk_size: Optional[int] = None            # chunk_sizes[level]; seq_len when unset
    alpha_floor: float = 0.0
    alpha_ceil: float = 1.0
    theta_floor: float = 0.0
    theta_ceil: float = F32_MAX
    error_clip: float = 0.0                     # error_clip_for_level(level); 0 = off
    m_norm_max: float = F32_MAX                 # max_m_norm(level)
    memory_layers: int = 1                      # 2 with "titans": the memory is a two-layer MLP per head
    memory_expansion_factor: int = 4            # its hidden size = factor * head_dim
    memory_activation: str = "gelu"             # "gelu", "silu", "relu"
    d_hidden: int = 0                           # MONETA / YAAD hidden size
    lp_p: float = 2.0                           # MONETA
    sign_sharpness: float = 10.0
    lambda_2: float = 0.0                       # MONETA and YAAD
    lq_q: float = 2.0
    delta: float = 1.0                          # YAAD: Huber threshold
    lambda_local: float = 0.0
    intermediate_size: int = 0                  # SwiGLU

    def __post_init__(self):
        if self.memory_rule not in RULES:
            raise ValueError(f"memory_rule {self.memory_rule!r}: expected one of {RULES}")
        if self.checkpoint_interval is not None and self.checkpoint_interval < 1:
            raise ValueError("checkpoint_interval must be > 0")
        if self.memory_activation not in ACTIVATIONS:
            raise ValueError(f"memory_activation {self.memory_activation!r}: expected one of {tuple(ACTIVATIONS)}")

    @property
    def is_mlp_mem(self):
        return self.memory_layers == 2 and self.memory_rule == "titans"


@dataclass
class GpuMemoryCache:
    """One of the reference's enum variants; `kind` is the variant's name."""
    kind: str
    k_mem: Optional[torch.Tensor] = None      # [bs*s, d] normalised
    v_mem: Optional[torch.Tensor] = None
    q_mem: Optional[torch.Tensor] = None      # [bs*s, d] normalised
    alpha: Optional[torch.Tensor] = None      # [bs*s]
    k_norms: Optional[torch.Tensor] = None
    q_norms: Optional[torch.Tensor] = None
    m_states: Optional[torch.Tensor] = None   # trajectory, checkpoints or chunk states (see the module text)
    theta: Optional[torch.Tensor] = None
    eta: Optional[torch.Tensor] = None
    s_states: Optional[torch.Tensor] = None
    checkpoint_interval: Optional[int] = None
    chunk_size: Optional[int] = None
    num_chunks: Optional[int] = None
    proxy: bool = False
    d_hidden: Optional[int] = None            # TitansMlp
    activation: Optional[int] = None
    w1_states: Optional[torch.Tensor] = None  # Mlp
    w2_states: Optional[torch.Tensor] = None
    w1_boundary: Optional[torch.Tensor] = None   # YAAD only: the memory at the start of the call
    w2_boundary: Optional[torch.Tensor] = None
    gate_buf: Optional[torch.Tensor] = None   # SwiGlu
    up_buf: Optional[torch.Tensor] = None
    fused_buf: Optional[torch.Tensor] = None
    cache_buf: Optional[torch.Tensor] = None
    group: Optional["LevelGroup"] = None      # the batch of levels this one ran in, and its place there
    group_index: int = 0

    def dgd_delta_norm(self, s, d, batch_size, num_heads):
        """|M k - v|_2 of the last token against the memory that token was written into
        (gpu_forward.rs:328-437): 0 for several heads, for Hebbian, and without tokens."""
        if num_heads > 1 or s == 0 or self.kind.startswith("Hebbian") or self.kind in ("TitansMlp", "Mlp", "SwiGlu"):
            return 0.0
        if self.proxy:   # only final states are kept (the TNT inner caches of a proxy level)
            return 0.0
        assert batch_size <= 1, "dgd_delta_norm reads batch slot 0 only"
        if self.kind.endswith("Chunkwise"):
            if not self.num_chunks:
                return 0.0
            slot = self.num_chunks - 1
        elif self.kind.endswith("Ckpt"):
            c = self.checkpoint_interval
            n_ckpt = (s + c - 1) // c + 1
            slot = n_ckpt - 2 if n_ckpt >= 2 else 0
        else:
            slot = s - 1
        out = torch.zeros(1, device=self.k_mem.device)
        D.call("dgd_delta_norm_cuda", self.m_states[0, slot].contiguous(), self.k_mem.reshape(-1, d)[s - 1].contiguous(),
               self.v_mem.reshape(-1, d)[s - 1].contiguous(), out, d)
        return float(out.item())

    def alpha_stats(self, alpha_floor):
        """gpu_forward.rs:440-503."""
        return None if self.alpha is None else GateStats.from_slice(self.alpha.cpu().numpy(), alpha_floor, True)

    def eta_stats(self):
        """gpu_forward.rs:505-564: only the Titans variants have a momentum gate."""
        return None if self.eta is None else GateStats.from_slice(self.eta.cpu().numpy(), 0.0, True)

    def theta_stats(self, theta_ceil):
        """gpu_forward.rs:566-623 (ThetaStats: the bound is a ceiling)."""
        return None if self.theta is None else GateStats.from_slice(self.theta.cpu().numpy(), theta_ceil, False)


@dataclass
class GateStats:
    """Distribution of one gate over the tokens of a forward pass (GateStats / ThetaStats,
    gpu_forward.rs:626-752): interpolated quantiles and the fraction of tokens on the configured bound."""
    count: int
    min: float
    max: float
    mean: float
    median: float
    p95: float
    p99: float
    frac_at_bound: float

    @staticmethod
    def from_slice(values, bound, bound_is_floor):
        v = np.sort(np.asarray(values, np.float32).ravel())
        n = v.size
        assert n > 0
        def quantile(p):
            rank = p * (n - 1.0)
            lo = int(np.floor(rank))
            hi = min(lo + 1, n - 1)
            frac = rank - lo
            return float(np.float32(float(v[lo]) * (1.0 - frac) + float(v[hi]) * frac))
        if bound_is_floor and bound > 0.0:
            at = int((v <= np.float32(bound * (1.0 + 1e-4))).sum())
        elif not bound_is_floor and bound < F32_MAX:
            at = int((v >= np.float32(bound * (1.0 - 1e-4))).sum())
        else:
            at = 0
        return GateStats(n, float(v[0]), float(v[-1]), float(v.sum(dtype=np.float32) / np.float32(n)),
                         quantile(0.5), quantile(0.95), quantile(0.99), at / n)


@dataclass
class LevelGrads:
    """GpuLevelGrads: gradients of one level's outer-loop parameters (overwritten by a backward)."""
    d_w_k_mem: torch.Tensor
    d_w_v_mem: torch.Tensor
    d_w_q_mem: torch.Tensor
    d_w_alpha: torch.Tensor
    d_b_alpha: torch.Tensor
    d_w_theta: torch.Tensor
    d_b_theta: torch.Tensor
    d_w_eta: torch.Tensor
    d_b_eta: torch.Tensor
    d_gate_proj: Optional[torch.Tensor] = None   # SwiGLU levels ([inter, d], [inter, d], [d, inter])
    d_up_proj: Optional[torch.Tensor] = None
    d_down_proj: Optional[torch.Tensor] = None

    @staticmethod
    def zeros(d, device="cuda", intermediate=0, cleared=True):
        """One buffer behind all tensors; cleared=False where a backward of every gate writes all of them."""
        sizes = [d * d] * 3 + [2 * d, 4] * 3
        flat = (torch.zeros if cleared else torch.empty)(sum(sizes), dtype=torch.float32, device=device)
        wk, wv, wq, wa, ba, wt, bt, we, be = flat.split(sizes)
        g = LevelGrads(wk.view(d, d), wv.view(d, d), wq.view(d, d), wa, ba[:1], wt, bt[:1], we, be[:1])
        z = lambda *sh: torch.zeros(*sh, dtype=torch.float32, device=device)
        if intermediate:
            g.d_gate_proj, g.d_up_proj, g.d_down_proj = z(intermediate, d), z(intermediate, d), z(d, intermediate)
        return g


@dataclass
class SwiGluLevelParams:
    """The parameters a SwiGLU level reads (GpuMemoryLevelParams gate_proj / up_proj / down_proj)."""
    gate_proj: torch.Tensor    # [intermediate, d]
    up_proj: torch.Tensor      # [intermediate, d]
    down_proj: torch.Tensor    # [d, intermediate]


def checkpoint_count(seq_len, c):
    """gpu_forward.rs:2885-2897: M_0, one slot per C-token boundary, the final state."""
    assert c > 0, "checkpoint_interval must be > 0"
    return 1 + sum(1 for t in range(seq_len) if (t + 1) % c == 0 or t + 1 == seq_len)


def segment_boundaries(seq_len, c):
    """gpu_backward.rs:1770-1782 -> [(t_start, t_end, ckpt_idx)]."""
    assert c > 0, "checkpoint_interval must be > 0"
    return [(t, min(t + c, seq_len), i) for i, t in enumerate(range(0, seq_len, c))]


def _new(*shape):
    return torch.empty(*shape, dtype=torch.float32, device="cuda")


def _zeros(*shape):
    return torch.zeros(*shape, dtype=torch.float32, device="cuda")


def _heads(cfg, t, bs, s):
    out = _new(bs * cfg.num_heads, s, cfg.head_dim)
    D.call("transpose_heads_f32_cuda", t, out, bs, s, cfg.num_heads, cfg.head_dim, 1)
    return out


def _tokens(cfg, t, bs, s):
    out = _new(bs * s, cfg.num_heads * cfg.head_dim)
    D.call("transpose_heads_f32_cuda", t, out, bs, s, cfg.num_heads, cfg.head_dim, 0)
    return out


def _gate_heads(cfg, g, bs, s):
    out = _new(bs * cfg.num_heads, s)
    D.call("broadcast_heads_f32_cuda", g, out, bs, s, cfg.num_heads)
    return out


def _sum_heads(cfg, g, bs, s):
    out = _new(bs * s)
    D.call("sum_heads_f32_cuda", g, out, bs, s, cfg.num_heads)
    return out


# ── levels as one batch ──────────────────────────────────────────────────────
# Levels that run the same rule with the same options on the same tokens are independent memories: their projections are
# one group of products, their glue one launch per step, and the rule one batch of levels * batch * heads chains.

class LevelGroup:
    """What a grouped forward leaves for the grouped backward: the head-major inputs of the rule, all levels stacked."""
    __slots__ = ("heads", "gates", "m_states", "s_states", "interval", "levels", "kind")

    def __init__(self, heads, gates, m_states, s_states, interval, levels, kind):
        self.heads, self.gates, self.m_states, self.s_states = heads, gates, m_states, s_states
        self.interval, self.levels, self.kind = interval, levels, kind


def group_key(cfg, level_params, d, bs):
    """Levels with equal keys can run as one batch; None: the level takes its own path."""
    if (cfg.memory_rule not in ("titans", "delta", "dgd") or cfg.memory_layers != 1 or d > 1024 or cfg.head_dim % 4
            or cfg.num_heads * cfg.head_dim != d or (cfg.proxy and cfg.memory_rule == "dgd")):
        return None
    # written out: nine tensors a level ahead of the first launch, where a call of _plain each costs half a launch
    lp, gates = level_params, 3 if cfg.memory_rule == "titans" else 2   # the momentum gate is not read without momentum
    f32, square = torch.float32, (d, d)
    for t in (lp.w_k, lp.w_v, lp.w_q):
        if t.dtype is not f32 or t.shape != square or not t.is_cuda or not t.is_contiguous() or t.data_ptr() & 15:
            return None
    for t in (lp.w_alpha, lp.w_theta, lp.w_eta)[:gates]:
        if t is None or t.dtype is not f32 or t.numel() != 2 * d or not t.is_cuda or not t.is_contiguous() or t.data_ptr() & 15:
            return None
    for t in (lp.b_alpha, lp.b_theta, lp.b_eta)[:gates]:
        if t is None or t.dtype is not f32 or t.numel() < 1 or not t.is_cuda or not t.is_contiguous():
            return None
    return (cfg.memory_rule, cfg.num_heads, cfg.head_dim, cfg.checkpoint_interval, cfg.proxy, cfg.chunk_size, cfg.error_clip,
            cfg.m_norm_max)


def _floats(t):
    """Contiguous floats on the device: what D.call asks of a buffer."""
    return isinstance(t, torch.Tensor) and t.dtype is torch.float32 and t.is_cuda and t.is_contiguous() and t.numel() > 0


def _plain(t, *shape):
    """_floats at a 16-byte boundary, which the grouped kernels read in 16-byte pieces; of this shape, if one is given."""
    return _floats(t) and not t.data_ptr() & 15 and (not shape or t.shape == shape)


def _grads_plain(g, d):
    """The gradients that backward_group writes, momentum gate included."""
    return (all(_plain(t, d, d) for t in (g.d_w_k_mem, g.d_w_v_mem, g.d_w_q_mem))
            and all(_floats(t) and t.numel() >= 2 * d for t in (g.d_w_alpha, g.d_w_theta, g.d_w_eta))
            and all(_floats(t) for t in (g.d_b_alpha, g.d_b_theta, g.d_b_eta)))


def _ptrs(tensors):
    return (ctypes.c_void_p * len(tensors))(*[t.data_ptr() for t in tensors])


def _bounds(cfgs):
    return (ctypes.c_float * (4 * len(cfgs)))(*[x for c in cfgs for x in (c.alpha_floor, c.alpha_ceil, c.theta_floor,
                                                                          c.theta_ceil)])


def _gate_params(lp, titans):
    """What level_group_inputs_f32_rocm takes of a level's gates; without momentum the last two are not read."""
    return (lp.w_alpha, lp.b_alpha, lp.w_theta, lp.b_theta) + ((lp.w_eta, lp.b_eta) if titans else (lp.w_alpha, lp.b_alpha))


def linear_group(op, a, b, c, m, n, k, bf16_mask=0):
    """Products of equal shape in one launch (linear_group_f32_rocm), 32 at a time."""
    if op == 1:
        lib.linear_group_f32_rocm(1, len(a), _ptrs(a), _ptrs(b), _ptrs(c), 0, m, n, k)
        return
    for i in range(0, len(a), 32):
        lib.linear_group_f32_rocm(op, len(a[i:i + 32]), _ptrs(a[i:i + 32]), _ptrs(b[i:i + 32]), _ptrs(c[i:i + 32]),
                                  (bf16_mask >> i) & 0xffffffff, m, n, k)


def product(op, a, b, c, m, n, k):
    """One product of any size (product_f32_rocm); operands as for op of linear_group, contiguous float32."""
    lib.product_f32_rocm(op, a.data_ptr(), b.data_ptr(), c.data_ptr(), m, n, k)


def forward_group(params, cfgs, embedded, contexts, s, d, bs):
    """gpu_memory_forward of a group of levels.  Returns (y [levels, bs*s, d], [cache per level])."""
    cfg, L = cfgs[0], len(cfgs)
    nh, hd = cfg.num_heads, cfg.head_dim
    n, B, dd = bs * s, bs * nh, hd * hd
    titans = cfg.memory_rule == "titans"
    proj = _new(3 * L, n, d)
    mem = list(proj.unbind(0))
    linear_group(0, [embedded] * (3 * L), [w for lp in params for w in (lp.w_k, lp.w_v, lp.w_q)], mem, n, d, d)
    gate = _new(5 * L, n)
    rows = list(gate.unbind(0))   # per level: k_norms, q_norms, alpha, theta, eta
    heads, gates = _new(3, L * B, s, hd), _new(3 if titans else 2, L * B, s)
    h0, g0 = heads.data_ptr(), gates.data_ptr()
    hs, gs = 4 * L * B * s * hd, 4 * L * B * s
    lib.level_group_inputs_f32_rocm(
        _ptrs([t for i, lp in enumerate(params) for t in (*mem[3 * i:3 * i + 3], *_gate_params(lp, titans), *rows[5 * i:5 * i + 5])]),
        _bounds(cfgs), L, h0, h0 + hs, h0 + 2 * hs, g0, g0 + gs, g0 + 2 * gs if titans else None, bs, s, nh, hd, 1e-8)
    initial = contexts[0]
    if L > 1:
        initial = _new(L * B, dd)
        lib.level_group_states_gather_rocm(_ptrs(contexts), L, initial.data_ptr(), B, dd)
    yh, clip, mx, C = _new(L * B, s, hd), cfg.error_clip, F32_MAX if cfg.memory_rule == "dgd" else cfg.m_norm_max, cfg.checkpoint_interval
    interval, form = 1, "" if C is None else "Ckpt"
    if C is not None:
        interval, slots = C, 1 + -(-s // C)
    elif cfg.proxy:
        interval, form = cfg.chunk_size or s, "Chunkwise"
        slots = -(-s // interval) + 1
    else:
        slots = s + 1
    m_states = _new(L * B, slots, dd)
    s_states = _new(L * B, slots, dd) if titans else None
    q = [h0, h0 + hs, h0 + 2 * hs, g0, g0 + gs]
    if titans:
        s_initial = _zeros(L * B, dd)   # by name: a tensor that is gone when the call starts is another thread's to take
        q += [g0 + 2 * gs, initial.data_ptr(), s_initial.data_ptr(), m_states.data_ptr(), s_states.data_ptr(), yh.data_ptr()]
    else:
        q += [initial.data_ptr(), m_states.data_ptr(), yh.data_ptr()]
    rule = "titans" if titans else "delta"
    if form == "Ckpt":
        getattr(lib, rule + "_forward_ckpt_batched_f32_rocm")(*q, s, hd, L * B, interval, clip, mx)
    elif form == "Chunkwise":
        getattr(lib, rule + "_chunkwise_forward_f32_cuda")(*q, s, hd, L * B, interval, clip, mx)
    else:
        getattr(lib, rule + "_forward_f32_cuda")(*q, s, hd, L * B, s, dd, clip, mx)
    # copy_final_m_batch + m_norm_clamp_batch_f32_cuda (gpu_forward.rs:2824, :1431)
    lib.level_group_states_final_rocm(m_states.data_ptr() + 4 * (slots - 1) * dd, slots * dd, _ptrs(contexts),
                                      (ctypes.c_float * L)(*[c.m_norm_max for c in cfgs]), L, B, dd)
    y = _new(L, n, d)
    lib.transpose_heads_f32_cuda(yh.data_ptr(), y.data_ptr(), L * bs, s, nh, hd, 0)
    kind = {"delta": "Delta", "titans": "Titans", "dgd": "DGD"}[cfg.memory_rule] + form
    group = LevelGroup(heads, gates, m_states, s_states, interval, L, kind)
    more = {"": {}, "Ckpt": dict(checkpoint_interval=C), "Chunkwise": dict(chunk_size=interval, num_chunks=slots - 1)}[form]
    mst = m_states.split(B)
    sst = s_states.split(B) if titans else [None] * L
    caches = [GpuMemoryCache(kind, k_mem=mem[3 * i], v_mem=mem[3 * i + 1], q_mem=mem[3 * i + 2], k_norms=rows[5 * i],
                             q_norms=rows[5 * i + 1], alpha=rows[5 * i + 2], theta=rows[5 * i + 3],
                             eta=rows[5 * i + 4] if titans else None, m_states=mst[i], s_states=sst[i], group=group,
                             group_index=i, **more) for i in range(L)]
    return y, caches


def backward_group(params, cfgs, caches, d_y, embedded, level_grads, s, d, bs, extra=()):
    """gpu_memory_backward of a whole group: every level sees the same d_y [bs*s, d].  extra: (gradient, weight, weight
    gradient) of further projections of `embedded`.  Fills the gradients and returns the sum of all input gradients."""
    cfg, L, g = cfgs[0], len(cfgs), caches[0].group
    nh, hd = cfg.num_heads, cfg.head_dim
    n, B, dd = bs * s, bs * nh, hd * hd
    titans = cfg.memory_rule == "titans"
    dyh = _new(L * B, s, hd)
    lib.level_group_heads_repeat_rocm(d_y.data_ptr(), dyh.data_ptr(), bs, s, nh, hd, L)
    dh, dg, d_init = _new(3, L * B, s, hd), _new(3 if titans else 2, L * B, s), _zeros(2, dd)
    h0, g0, e0, f0, i0 = (t.data_ptr() for t in (g.heads, g.gates, dh, dg, d_init))
    hs, gs = 4 * L * B * s * hd, 4 * L * B * s
    clip, mx = cfg.error_clip, F32_MAX if cfg.memory_rule == "dgd" else cfg.m_norm_max
    if titans:
        args = [h0, h0 + hs, h0 + 2 * hs, g0, g0 + gs, g0 + 2 * gs, g.m_states.data_ptr(), g.s_states.data_ptr(), dyh.data_ptr(),
                e0, e0 + hs, e0 + 2 * hs, f0, f0 + gs, f0 + 2 * gs, i0, i0 + 4 * dd]
    else:
        args = [h0, h0 + hs, h0 + 2 * hs, g0, g0 + gs, g.m_states.data_ptr(), dyh.data_ptr(), e0, e0 + hs, e0 + 2 * hs, f0, f0 + gs, i0]
    rule = "titans" if titans else "delta"
    fn = rule + ("_chunkwise_backward_f32_cuda" if g.kind.endswith("Chunkwise") else "_backward_ckpt_f32_rocm")
    getattr(lib, fn)(*args, s, hd, L * B, g.interval, clip, mx)
    raw = list(_new(3 * L, n, d).unbind(0))   # d_k, d_v, d_q of the raw projections, per level
    ptrs = []
    for i, (c, lg) in enumerate(zip(caches, level_grads)):
        eta = c.eta if titans else c.alpha     # not read without the momentum gate
        ptrs += (c.k_mem, c.v_mem, c.q_mem, c.k_norms, c.q_norms, c.alpha, c.theta, eta, *raw[3 * i:3 * i + 3], lg.d_w_alpha,
                 lg.d_b_alpha, lg.d_w_theta, lg.d_b_theta, lg.d_w_eta, lg.d_b_eta)
    lib.level_group_grads_f32_rocm(_ptrs(ptrs), _bounds(cfgs), L, e0, e0 + hs, e0 + 2 * hs, f0, f0 + gs,
                                   f0 + 2 * gs if titans else None, bs, s, nh, hd, 1e-8)
    up = raw + [x for x, _, _ in extra]
    linear_group(2, up, [embedded] * len(up),
                 [w for lg in level_grads for w in (lg.d_w_k_mem, lg.d_w_v_mem, lg.d_w_q_mem)] + [w for _, _, w in extra], d, d, n)
    d_embedded = _new(n, d)
    linear_group(1, up, [w for lp in params for w in (lp.w_k, lp.w_v, lp.w_q)] + [w for _, w, _ in extra], [d_embedded], n, d, d)
    return d_embedded


def gpu_memory_forward(level_params: MemoryLevelParams, cfg: LevelConfig, embedded, context_m, s, d, batch_size):
    """embedded [bs*s, d]; context_m [bs*nh, hd*hd]: the level's carried memory per (batch, head), read as the
    initial state and overwritten with the final one.  Returns (y [bs*s, d], GpuMemoryCache)."""
    lp, bs, nh, hd = level_params, batch_size, cfg.num_heads, cfg.head_dim
    assert nh * hd == d, "num_heads * head_dim must equal d"
    n, B, dd = bs * s, bs * nh, hd * hd
    assert tuple(embedded.shape) == (n, d)
    rule = cfg.memory_rule
    if rule == "swiglu":   # stateless: no projections, no memory (gpu_forward.rs:1705-1727)
        inter = cfg.intermediate_size
        bufs = [_new(n, inter) for _ in range(4)]
        y = _new(n, d)
        D.call("swiglu_forward_f32_cuda_dd", embedded, lp.gate_proj, lp.up_proj, lp.down_proj, y, *bufs, n, d, inter)
        return y, GpuMemoryCache("SwiGlu", gate_buf=bufs[0], up_buf=bufs[1], fused_buf=bufs[2], cache_buf=bufs[3])
    if cfg.is_mlp_mem and (cfg.checkpoint_interval is not None or cfg.proxy):
        raise ValueError("MLP memory (memory_layers >= 2) supports neither checkpointing nor the proxy strategy")
    if rule in ("moneta", "yaad"):
        if cfg.checkpoint_interval is not None:
            raise ValueError(f"checkpointed forward is not supported for {rule}: use checkpoint_interval=None")
        if bs != 1:
            raise ValueError(f"{rule} forward with batch_size > 1 is not supported")
    elif not cfg.is_mlp_mem:
        assert tuple(context_m.shape) == (B, dd)
    if group_key(cfg, lp, d, bs) is not None and _plain(embedded, n, d) and _plain(context_m, B, dd):
        y, caches = forward_group([lp], [cfg], embedded, [context_m], s, d, bs)
        return y[0], caches[0]
    k_mem, v_mem, q_mem = embedded @ lp.w_k.t(), embedded @ lp.w_v.t(), embedded @ lp.w_q.t()
    k_norms, q_norms = _new(n), _new(n)
    D.call("l2_normalize_rows_f32_cuda", k_mem, k_norms, n, d, 1e-8)
    D.call("l2_normalize_rows_f32_cuda", q_mem, q_norms, n, d, 1e-8)
    alpha, theta = _new(n), _new(n)
    D.call("gate_compute_cuda", k_mem, v_mem, lp.w_alpha, lp.b_alpha, alpha, n, d, 0)
    D.call("gate_compute_cuda", k_mem, v_mem, lp.w_theta, lp.b_theta, theta, n, d, 1)
    if cfg.alpha_floor > 0.0 or cfg.alpha_ceil < 1.0:
        D.call("clamp_f32_cuda", alpha, n, cfg.alpha_floor, cfg.alpha_ceil)
    if cfg.theta_floor > 0.0 or cfg.theta_ceil < F32_MAX:
        D.call("clamp_f32_cuda", theta, n, cfg.theta_floor, cfg.theta_ceil)
    common = dict(k_mem=k_mem, v_mem=v_mem, q_mem=q_mem, alpha=alpha, k_norms=k_norms, q_norms=q_norms)
    if rule in ("moneta", "yaad"):
        return _mlp_forward(cfg, context_m, theta, common, s, d)
    kh, vh, qh = (_heads(cfg, t, bs, s) for t in (k_mem, v_mem, q_mem))
    ah, th = _gate_heads(cfg, alpha, bs, s), _gate_heads(cfg, theta, bs, s)
    eta = eh = None
    if rule == "titans":   # compute_eta, gpu_forward.rs:2866
        eta = _new(n)
        D.call("gate_compute_cuda", k_mem, v_mem, lp.w_eta, lp.b_eta, eta, n, d, 0)
        eh = _gate_heads(cfg, eta, bs, s)
    yh = _new(B, s, hd)
    clip, mx, C = cfg.error_clip, cfg.m_norm_max, cfg.checkpoint_interval
    s_states = None
    if cfg.is_mlp_mem:
        # the memory of a head is {W1, b1, W2, b2} packed; the kernel projects per token, so the carried state
        # needs no clamp afterwards (gpu_forward.rs:1473-1510)
        d_h = cfg.memory_expansion_factor * hd
        n_state = 2 * hd * d_h + d_h + hd
        assert tuple(context_m.shape) == (B, n_state)
        act = ACTIVATIONS[cfg.memory_activation]
        m_states, s_states = _new(B, s + 1, n_state), _new(B, s + 1, n_state)
        D.call("titans_mlp_forward_f32_cuda", kh, vh, qh, ah, th, eh, context_m, _zeros(B, n_state), m_states, s_states,
               yh, s, hd, d_h, B, s * hd, (s + 1) * n_state, act, mx)
        context_m.copy_(m_states[:, -1])
        cache = GpuMemoryCache("TitansMlp", theta=theta, eta=eta, m_states=m_states, s_states=s_states, d_hidden=d_h,
                               activation=act, **common)
        return _tokens(cfg, yh, bs, s), cache
    if C is not None:
        n_ck = checkpoint_count(s, C)
        m_states = _new(B, n_ck, dd)
        if rule == "titans":
            s_states = _new(B, n_ck, dd)
            D.call("titans_forward_ckpt_batched_f32_rocm", kh, vh, qh, ah, th, eh, context_m, _zeros(B, dd), m_states,
                   s_states, yh, s, hd, B, C, clip, mx)
        elif rule == "hebbian":
            flat = lambda t: t.view(-1)
            for b in range(B):   # single-chain entry point, as the reference calls it (gpu_forward.rs:1669)
                D.call("hebbian_forward_ckpt_f32_cuda", flat(kh)[b * s * hd:], flat(vh)[b * s * hd:],
                       flat(qh)[b * s * hd:], flat(ah)[b * s:], flat(context_m)[b * dd:],
                       flat(m_states)[b * n_ck * dd:], flat(yh)[b * s * hd:], s, hd, C)
        else:   # DGD: Delta without the per-token projection (core/kernels/dgd_forward.cu:6-11)
            D.call("delta_forward_ckpt_batched_f32_rocm", kh, vh, qh, ah, th, context_m, m_states, yh, s, hd, B, C,
                   clip, F32_MAX if rule == "dgd" else mx)
        kind = {"delta": "DeltaCkpt", "titans": "TitansCkpt", "hebbian": "HebbianCkpt", "dgd": "DGDCkpt"}[rule]
        cache = GpuMemoryCache(kind, theta=None if rule == "hebbian" else theta, eta=eta, m_states=m_states,
                               s_states=s_states, checkpoint_interval=C, **common)
    elif cfg.proxy and rule in ("delta", "titans"):
        cs = cfg.chunk_size or s
        nc = (s + cs - 1) // cs
        m_states = _new(B, nc + 1, dd)
        if rule == "titans":
            s_states = _new(B, nc + 1, dd)
            D.call("titans_chunkwise_forward_f32_cuda", kh, vh, qh, ah, th, eh, context_m, _zeros(B, dd), m_states,
                   s_states, yh, s, hd, B, cs, clip, mx)
        else:
            D.call("delta_chunkwise_forward_f32_cuda", kh, vh, qh, ah, th, context_m, m_states, yh, s, hd, B, cs,
                   clip, mx)
        cache = GpuMemoryCache("TitansChunkwise" if rule == "titans" else "DeltaChunkwise", theta=theta, eta=eta,
                               m_states=m_states, s_states=s_states, chunk_size=cs, num_chunks=nc, **common)
    else:
        m_states = _new(B, s + 1, dd)
        if rule == "titans":
            s_states = _new(B, s + 1, dd)
            D.titans_forward_dd(kh, vh, qh, ah, th, eh, context_m, _zeros(B, dd), m_states, s_states, yh, s, hd, B,
                                s, dd, clip, mx)
        elif rule == "hebbian":
            D.call("hebbian_forward_f32_cuda", kh, vh, qh, ah, context_m, m_states, yh, s, hd, B, s, dd)
        elif rule == "dgd":
            D.call("dgd_forward_f32_cuda", kh, vh, qh, ah, th, context_m, m_states, yh, s, hd, B, s, dd, clip)
        else:
            D.call("delta_forward_f32_cuda", kh, vh, qh, ah, th, context_m, m_states, yh, s, hd, B, s, dd, clip, mx)
        kind = {"delta": "Delta", "titans": "Titans", "hebbian": "Hebbian", "dgd": "DGD"}[rule]
        cache = GpuMemoryCache(kind, theta=None if rule == "hebbian" else theta, eta=eta, m_states=m_states,
                               s_states=s_states, **common)
    # copy_final_m_batch + m_norm_clamp_batch_f32_cuda (gpu_forward.rs:2824, :1431)
    context_m.copy_(m_states[:, -1])
    D.call("m_norm_clamp_batch_f32_cuda", context_m, hd, B, mx)
    return _tokens(cfg, yh, bs, s), cache


def _mlp_forward(cfg, context_m, theta, common, s, d):
    """MONETA / YAAD: an MLP memory at model width, one sequence; context_m = [W1 (dh x d) | W2 (d x dh)]
    (gpu_forward.rs:1729-1852)."""
    dh = cfg.d_hidden
    w1_size, w2_size = dh * d, d * dh
    flat = context_m.view(-1)
    if flat.numel() < w1_size + w2_size:
        raise ValueError(f"{cfg.memory_rule}: context_m too small ({flat.numel()} elements) for [W1|W2] = "
                         f"{w1_size + w2_size} (d_hidden={dh}, d={d})")
    w1, w2 = flat[:w1_size], flat[w1_size:w1_size + w2_size]
    w1_states, w2_states, y = _new(s + 1, w1_size), _new(s + 1, w2_size), _new(s, d)
    c = common
    b1 = b2 = None
    if cfg.memory_rule == "yaad":   # the memory at the start of the call anchors the local retention
        b1, b2 = w1.clone(), w2.clone()
        D.call("mlp_forward_huber_f32_cuda", c["k_mem"], c["v_mem"], c["q_mem"], c["alpha"], theta, w1, w2, b1, b2,
               w1_states, w2_states, y, s, d, dh, cfg.delta, cfg.lambda_local, cfg.lambda_2)
    else:
        D.call("mlp_forward_lp_f32_cuda", c["k_mem"], c["v_mem"], c["q_mem"], c["alpha"], theta, w1, w2, w1_states,
               w2_states, y, s, d, dh, cfg.lp_p, cfg.sign_sharpness, cfg.lambda_2, cfg.lq_q)
    w1.copy_(w1_states[s])
    w2.copy_(w2_states[s])
    return y, GpuMemoryCache("Mlp", theta=theta, w1_states=w1_states, w2_states=w2_states, w1_boundary=b1,
                             w2_boundary=b2, **common)


def gpu_memory_backward(level_params: MemoryLevelParams, cfg: LevelConfig, mem_cache: GpuMemoryCache, d_y, embedded,
                        level_grads: LevelGrads, s, d, batch_size):
    """d_y, embedded [bs*s, d].  Writes the level's parameter gradients into level_grads and returns
    d_embedded [bs*s, d]."""
    c, bs, nh, hd = mem_cache, batch_size, cfg.num_heads, cfg.head_dim
    n, B, dd = bs * s, bs * nh, hd * hd
    kind = c.kind
    if kind == "SwiGlu":   # direct weight gradients, d_x returned (gpu_backward.rs:1736-1760)
        inter = cfg.intermediate_size
        d_x = _new(n, d)
        D.call("swiglu_backward_f32_cuda_dd", d_y, embedded, level_params.gate_proj, level_params.up_proj,
               level_params.down_proj, c.fused_buf, c.gate_buf, c.up_buf, c.cache_buf, d_x, level_grads.d_gate_proj,
               level_grads.d_up_proj, level_grads.d_down_proj, n, d, inter)
        return d_x
    if kind == "Mlp":
        return _mlp_backward(level_params, cfg, c, d_y, embedded, level_grads, s, d, bs)
    if (c.group is not None and c.group.levels == 1 and group_key(cfg, level_params, d, bs) is not None and _plain(d_y)
            and d_y.numel() == n * d and _plain(embedded, n, d) and _grads_plain(level_grads, d)):
        return backward_group([level_params], [cfg], [c], d_y, embedded, [level_grads], s, d, bs)
    has_theta, has_eta = not kind.startswith("Hebbian"), kind.startswith("Titans")
    dyh = _heads(cfg, d_y, bs, s)
    kh, vh, qh = (_heads(cfg, t, bs, s) for t in (c.k_mem, c.v_mem, c.q_mem))
    ah = _gate_heads(cfg, c.alpha, bs, s)
    th = _gate_heads(cfg, c.theta, bs, s) if has_theta else None
    eh = _gate_heads(cfg, c.eta, bs, s) if has_eta else None
    dkh, dvh, dqh = _zeros(B, s, hd), _zeros(B, s, hd), _zeros(B, s, hd)
    dah, dth, deh = _zeros(B, s), _zeros(B, s), _zeros(B, s)
    d_m0, d_s0 = _zeros(dd), _zeros(dd)
    clip, mx = cfg.error_clip, cfg.m_norm_max
    if kind in ("Delta", "DGD"):   # a trajectory is a checkpoint per token; the DGD forward ran without the projection
        D.call("delta_backward_ckpt_f32_rocm", kh, vh, qh, ah, th, c.m_states, dyh, dkh, dvh, dqh, dah, dth, d_m0, s, hd,
               B, 1, clip, F32_MAX if kind == "DGD" else mx)
    elif kind == "Titans":
        D.call("titans_backward_ckpt_f32_rocm", kh, vh, qh, ah, th, eh, c.m_states, c.s_states, dyh, dkh, dvh, dqh, dah,
               dth, deh, d_m0, d_s0, s, hd, B, 1, clip, mx)
    elif kind == "DeltaChunkwise":
        D.call("delta_chunkwise_backward_f32_cuda", kh, vh, qh, ah, th, c.m_states, dyh, dkh, dvh, dqh, dah, dth,
               d_m0, s, hd, B, c.chunk_size, clip, mx)
    elif kind == "TitansChunkwise":
        D.call("titans_chunkwise_backward_f32_cuda", kh, vh, qh, ah, th, eh, c.m_states, c.s_states, dyh, dkh, dvh,
               dqh, dah, dth, deh, d_m0, d_s0, s, hd, B, c.chunk_size, clip, mx)
    elif kind == "Hebbian":
        flat = lambda t: t.view(-1)
        for b in range(B):   # single-chain entry point, one call per head (gpu_backward.rs:913-930)
            D.call("hebbian_backward_f32_cuda", flat(kh)[b * s * hd:], flat(vh)[b * s * hd:], flat(qh)[b * s * hd:],
                   flat(ah)[b * s:], flat(c.m_states)[b * (s + 1) * dd:], flat(dyh)[b * s * hd:],
                   flat(dkh)[b * s * hd:], flat(dvh)[b * s * hd:], flat(dqh)[b * s * hd:], flat(dah)[b * s:], d_m0,
                   s, hd)
    elif kind in ("DeltaCkpt", "DGDCkpt"):
        # one call walks the segments in reverse (the host loop delta_backward_checkpointed, gpu_backward.rs:1791);
        # the DGD replay leaves the projection off as its forward did (:1156-1161)
        D.call("delta_backward_ckpt_f32_rocm", kh, vh, qh, ah, th, c.m_states, dyh, dkh, dvh, dqh, dah, dth, d_m0, s,
               hd, B, c.checkpoint_interval, clip, F32_MAX if kind == "DGDCkpt" else mx)
    elif kind == "TitansMlp":
        n_state = c.m_states.shape[-1]
        D.call("titans_mlp_backward_f32_cuda", kh, vh, qh, ah, th, eh, c.m_states, c.s_states, dyh, dkh, dvh, dqh, dah,
               dth, deh, _zeros(n_state), _zeros(n_state), s, hd, c.d_hidden, B, s * hd, (s + 1) * n_state,
               c.activation, mx)
    elif kind == "TitansCkpt":
        D.call("titans_backward_ckpt_f32_rocm", kh, vh, qh, ah, th, eh, c.m_states, c.s_states, dyh, dkh, dvh, dqh,
               dah, dth, deh, d_m0, d_s0, s, hd, B, c.checkpoint_interval, clip, mx)
    elif kind == "HebbianCkpt":
        _hebbian_backward_checkpointed(kh, vh, qh, ah, c.m_states, dyh, dkh, dvh, dqh, dah, s, hd,
                                       c.checkpoint_interval, B)
    else:
        raise ValueError(f"gpu_memory_backward: unsupported cache variant {kind}")
    d_alpha = _sum_heads(cfg, dah, bs, s)
    d_theta = _sum_heads(cfg, dth, bs, s) if has_theta else None
    d_eta = _sum_heads(cfg, deh, bs, s) if has_eta else None
    # straight-through clamps: no gradient where the gate sat on a bound
    if cfg.alpha_floor > 0.0 or cfg.alpha_ceil < 1.0:
        D.call("theta_clamp_mask_cuda", c.alpha, d_alpha, n, cfg.alpha_floor, cfg.alpha_ceil)
    if has_theta and (cfg.theta_floor > 0.0 or cfg.theta_ceil < F32_MAX):
        D.call("theta_clamp_mask_cuda", c.theta, d_theta, n, cfg.theta_floor, cfg.theta_ceil)
    d_k, d_v, d_q = (_tokens(cfg, t, bs, s) for t in (dkh, dvh, dqh))
    return accumulate_projection_grads(level_params, embedded, c, d_k, d_v, d_q, d_alpha, d_theta, d_eta, level_grads,
                                       s, d, bs)


def _mlp_backward(level_params, cfg, c, d_y, embedded, level_grads, s, d, bs):
    """MONETA (L2 retention only: lq_q = 2) / YAAD backward at model width, one sequence
    (gpu_backward.rs:1635-1733).  As in the reference the gradients of the initial W1, W2 are computed and
    not used."""
    if bs != 1:
        raise ValueError("MLP memory backward with batch_size > 1 is not supported")
    dh = cfg.d_hidden
    d_k, d_v, d_q = _zeros(s, d), _zeros(s, d), _zeros(s, d)
    d_alpha, d_theta = _zeros(s), _zeros(s)
    d_w1, d_w2 = _zeros(dh * d), _zeros(d * dh)
    if (c.w1_boundary is None) != (c.w2_boundary is None):
        raise ValueError("MLP backward: W1 and W2 boundaries must both be present (YAAD) or both absent (MONETA)")
    if c.w1_boundary is not None:
        D.call("mlp_backward_huber_f32_cuda", c.k_mem, c.v_mem, c.q_mem, c.alpha, c.theta, c.w1_states, c.w2_states,
               c.w1_boundary, c.w2_boundary, d_y, d_k, d_v, d_q, d_alpha, d_theta, d_w1, d_w2, s, d, dh, cfg.delta,
               cfg.lambda_local, cfg.lambda_2)
    else:
        if abs(cfg.lq_q - 2.0) >= 1e-6:
            raise ValueError(f"MONETA backward only supports lq_q=2.0 (L2 retention); got {cfg.lq_q}")
        D.call("mlp_backward_lp_f32_cuda", c.k_mem, c.v_mem, c.q_mem, c.alpha, c.theta, c.w1_states, c.w2_states, d_y,
               d_k, d_v, d_q, d_alpha, d_theta, d_w1, d_w2, s, d, dh, cfg.lp_p, cfg.sign_sharpness, cfg.lambda_2,
               cfg.lq_q)
    if cfg.alpha_floor > 0.0 or cfg.alpha_ceil < 1.0:
        D.call("theta_clamp_mask_cuda", c.alpha, d_alpha, s, cfg.alpha_floor, cfg.alpha_ceil)
    if cfg.theta_floor > 0.0 or cfg.theta_ceil < F32_MAX:
        D.call("theta_clamp_mask_cuda", c.theta, d_theta, s, cfg.theta_floor, cfg.theta_ceil)
    return accumulate_projection_grads(level_params, embedded, c, d_k, d_v, d_q, d_alpha, d_theta, None, level_grads, s,
                                       d, 1)


def _hebbian_backward_checkpointed(kh, vh, qh, ah, m_ckpt, dyh, dkh, dvh, dqh, dah, s, hd, c, B):
    """hebbian_backward_checkpointed (gpu_backward.rs:1967-2035): per segment, last first, replay the
    trajectory of every chain from its checkpoint, then the batched segment backward seeded with the
    state gradient of the segment after it."""
    dd = hd * hd
    n_ck = checkpoint_count(s, c)
    seg_max = min(c, s)
    local_m, local_y = _new(B, seg_max + 1, dd), _new(B, seg_max, hd)
    seed, out = _zeros(B, dd), _zeros(B, dd)
    flat = lambda t: t.view(-1)
    for t0, t1, ci in reversed(segment_boundaries(s, c)):
        seg = t1 - t0
        lm = local_m if seg == seg_max else _new(B, seg + 1, dd)
        ly = local_y if seg == seg_max else _new(B, seg, hd)
        D.call("hebbian_forward_f32_cuda", flat(kh)[t0 * hd:], flat(vh)[t0 * hd:], flat(qh)[t0 * hd:], flat(ah)[t0:],
               flat(m_ckpt)[ci * dd:], lm, ly, seg, hd, B, s, n_ck * dd)
        out.zero_()
        D.call("hebbian_backward_segment_f32_cuda", kh, vh, qh, ah, lm, dyh, seed, dkh, dvh, dqh, dah, out, t0, t1, hd,
               B, s)
        seed.copy_(out)


def accumulate_projection_grads(level_params, embedded, cache, d_k_mem, d_v_mem, d_q_mem, d_alpha, d_theta, d_eta,
                                level_grads, s, d, batch_size):
    """gpu_backward.rs:2047-2117.  As in the reference the gate gradients reach the gate weights and biases
    only; k_mem and v_mem receive nothing through the gates."""
    lp, c, g = level_params, cache, level_grads
    n = batch_size * s
    d_k_raw, d_q_raw = _new(n, d), _new(n, d)
    D.call("l2_normalize_backward_f32_cuda", d_k_mem, c.k_mem, c.k_norms, d_k_raw, n, d, 1e-8)
    D.call("l2_normalize_backward_f32_cuda", d_q_mem, c.q_mem, c.q_norms, d_q_raw, n, d, 1e-8)
    torch.mm(d_k_raw.t(), embedded, out=g.d_w_k_mem)
    torch.mm(d_v_mem.t(), embedded, out=g.d_w_v_mem)
    torch.mm(d_q_raw.t(), embedded, out=g.d_w_q_mem)
    d_embedded = d_k_raw @ lp.w_k
    d_embedded.addmm_(d_v_mem, lp.w_v)
    d_embedded.addmm_(d_q_raw, lp.w_q)
    z = d_alpha   # placeholder for the absent gates: not read when the has_* flag is 0
    D.call("gate_backward_cuda", d_alpha, c.alpha, d_theta if d_theta is not None else z,
           c.theta if c.theta is not None else z, d_eta if d_eta is not None else z,
           c.eta if c.eta is not None else z, c.k_mem, c.v_mem, g.d_w_alpha, g.d_b_alpha, g.d_w_theta, g.d_b_theta,
           g.d_w_eta, g.d_b_eta, n, d, int(d_theta is not None), int(d_eta is not None))
    return d_embedded
