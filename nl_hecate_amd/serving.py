"""Host mirror of the reference's cached generation path on device buffers:
GpuKVCache (core/src/gpu_forward.rs:2979-3147), gpu_prefill_forward (:3160-3312), DecodeWorkspace
(:3321-3362) and gpu_single_token_forward (:3377-3492).

Prefill runs the full forward over the prompt, fills the bf16 K/V cache and returns the logits of the
last position; a decode step embeds one token, appends its K and V, attends over the cache
(swa_single_token_cuda), runs every memory level with seq_len = 1 on the carried context memory
(active levels: the level step of memory_level.py; frozen levels: a read of the memory), combines the
levels, gates the attention output, projects and unembeds.  Every step is a call into
libnl_hecate_rocm.so or a torch matmul in the place of the reference's cuBLAS calls; the only transfers are
the token ids in and the logits out, as in the reference.
"""
import ctypes
import operator
from dataclasses import dataclass, field
from typing import List

import numpy as np
import torch

from . import dispatch as D
from . import ffi
from .cms import ContextState, Pulse
from .ffi import lib
from .mag_layer import MemoryLevelParams
from .memory_level import F32_MAX, LevelConfig, _gate_params, _plain, _ptrs, gpu_memory_forward, group_key, linear_group


def _new(*shape, dtype=torch.float32):
    return torch.empty(*shape, dtype=dtype, device="cuda")


def _zeros(*shape, dtype=torch.float32):
    return torch.zeros(*shape, dtype=dtype, device="cuda")


def host_ids(ids):
    """Token ids as int32 on the host.  Whatever does not fit is refused, not wrapped; other numbers go through int()."""
    if isinstance(ids, torch.Tensor):
        ids = ids.cpu()
    elif isinstance(ids, (list, tuple)) and ids and isinstance(ids[0], torch.Tensor):
        ids = [int(t) for t in ids]
    a = np.asarray(ids)
    if a.dtype.kind not in "iu":
        a = np.array([int(t) for t in a], dtype=np.int64 if not a.size else None)
    if a.dtype.itemsize >= 4 and a.dtype != np.int32 and a.size and not -2 ** 31 <= a.min() <= a.max() < 2 ** 31:
        raise RuntimeError("token id cannot be converted to int32 without overflow")
    return a.astype(np.int32, copy=False)


@dataclass
class GpuMAGParams:
    """The tensors the generation path reads (GpuMAGParams: swa block + levels)."""
    w_embed: torch.Tensor      # [vocab, d]
    w_q: torch.Tensor          # [d, d]
    w_k: torch.Tensor
    w_v: torch.Tensor
    w_o: torch.Tensor
    w_unembed: torch.Tensor    # [d, vocab]
    levels: List[MemoryLevelParams] = field(default_factory=list)


@dataclass
class ServeConfig:
    """What the two functions read from MAGConfig."""
    d_model: int
    vocab_size: int
    num_heads: int
    head_dim: int
    window_size: int
    seq_len: int                    # prompt length of a prefill
    levels: List[LevelConfig]       # one per CMS level (cfg.k = len(levels))
    n_persistent: int = 0
    decode_tokens: int = 2048       # prefill sizes the cache for the prompt plus this many decode tokens
    residual: bool = False          # the reference's cached-generation path refuses residual = true (:3175, :3392)

    @property
    def k(self):
        return len(self.levels)


class GpuKVCache:
    """bf16 K and V of every position so far, [max_len, d] each, with a conversion scratch sized once."""

    def __init__(self, max_len, d, scratch_tokens):
        self.k_cache_bf16, self.v_cache_bf16 = _zeros(2, max_len, d, dtype=torch.bfloat16).unbind(0)
        self.len, self.max_len, self.d = 0, max_len, d
        self._scratch_k, self._scratch_v = _new(2, scratch_tokens * d, dtype=torch.bfloat16).unbind(0)

    def append_f32(self, k_f32, v_f32, n_tokens):
        """:3017-3053: convert into the scratch, copy behind the filled positions."""
        if self.len + n_tokens > self.max_len:
            raise OverflowError(f"KV cache overflow: {self.len} + {n_tokens} > {self.max_len}")
        total = n_tokens * self.d
        if total > self._scratch_k.numel():
            raise ValueError(f"append_f32: n_tokens*d={total} exceeds scratch buffer size {self._scratch_k.numel()}")
        D.call("f32_to_bf16_cuda", k_f32, self._scratch_k, total)
        D.call("f32_to_bf16_cuda", v_f32, self._scratch_v, total)
        self.k_cache_bf16.view(-1)[self.len * self.d:self.len * self.d + total].copy_(self._scratch_k[:total])
        self.v_cache_bf16.view(-1)[self.len * self.d:self.len * self.d + total].copy_(self._scratch_v[:total])
        self.len += n_tokens

    def _project_persistent(self, persistent_tokens, w_k, w_v, n_persistent, d):
        if d != self.d:
            raise ValueError(f"persistent tokens: caller d={d} != cache d={self.d}")
        npd = n_persistent * d
        if persistent_tokens.numel() < npd:
            raise ValueError(f"persistent_tokens has {persistent_tokens.numel()} < n_persistent*d={npd} elements")
        p = persistent_tokens.reshape(-1)[:npd].view(n_persistent, d)
        pk, pv = (p @ w_k.t()).contiguous(), (p @ w_v.t()).contiguous()
        D.call("f32_to_bf16_cuda", pk, self.k_cache_bf16, npd)
        D.call("f32_to_bf16_cuda", pv, self.v_cache_bf16, npd)

    def prepopulate_persistent(self, persistent_tokens, w_k, w_v, n_persistent, d):
        """:3055-3099: positions [0, n_persistent) = projections of the persistent tokens; empty cache only."""
        if n_persistent == 0:
            return
        if n_persistent > self.max_len:
            raise OverflowError(f"KV cache too small for {n_persistent} persistent tokens")
        if self.len != 0:
            raise RuntimeError("prepopulate_persistent must be called on an empty cache")
        self._project_persistent(persistent_tokens, w_k, w_v, n_persistent, d)
        self.len = n_persistent

    def refresh_persistent(self, persistent_tokens, w_k, w_v, n_persistent, d):
        """:3101-3141: the same projection after an optimizer step; the length does not change."""
        if n_persistent == 0:
            return
        if self.len < n_persistent:
            raise RuntimeError(f"cache len {self.len} < n_persistent {n_persistent}")
        self._project_persistent(persistent_tokens, w_k, w_v, n_persistent, d)

    def reset(self):
        self.len = 0


class DecodeWorkspace:
    """Buffers of one decode step, allocated once (:3321-3362)."""

    def __init__(self, d, v):
        self.d_input = _zeros(1, dtype=torch.int32)
        self.embedded = _zeros(1, d)
        self.q_bf16 = _zeros(1, d, dtype=torch.bfloat16)
        self.attn_out_bf16 = _zeros(1, d, dtype=torch.bfloat16)
        self.attn_out = _zeros(1, d)
        self.y_combined, self.gate, self.gated_out = _zeros(1, d), _zeros(1, d), _zeros(1, d)
        self.logits_gpu = _zeros(1, v)
        # of the library's one-call step: intermediates of its launches, its argument blocks, the logits where the host
        # reads them
        self.work = _new(0)
        self.plans = {}
        self.logits_host = torch.empty(v, dtype=torch.float32, pin_memory=True)

    def __getstate__(self):
        """Copied and saved without what holds addresses."""
        return {n: t for n, t in self.__dict__.items() if n not in ("work", "plans")}

    def __setstate__(self, state):
        host = state.get("logits_host")   # absent from what was saved before the one-call step
        self.__dict__.update(state, work=_new(0), plans={}, logits_host=(
            torch.empty(state["logits_gpu"].shape[-1]) if host is None else host).pin_memory())

    def written(self):
        """What the one-call step writes besides the logits on the host, in the order of its argument block."""
        return (self.embedded, self.q_bf16, self.attn_out_bf16, self.attn_out, self.y_combined, self.gate, self.gated_out,
                self.logits_gpu)

    def work_for(self, floats):
        if self.work.numel() < floats:
            self.work = _new(floats)
            self.plans.clear()   # they hold the old buffer's address
        return self.work


def _keys_fit(cfg, pos):
    """The one-call step merges its slices of 128 keys in 64 KB of LDS: model width + slices * heads floats."""
    keys = min(pos + 1, cfg.window_size + cfg.n_persistent)
    return cfg.d_model + -(-keys // 128) * cfg.num_heads <= 16384


# level_rule of decode_token_rocm; a Titans level starts every call with zero momentum, so its one-token step is Delta's
_LEVEL_TENSORS = operator.attrgetter("w_k", "w_v", "w_q", "w_alpha", "b_alpha", "w_theta", "b_theta")
_LEVEL_OPTIONS = operator.attrgetter("memory_rule", "memory_layers", "num_heads", "head_dim", "alpha_floor", "alpha_ceil",
                                     "theta_floor", "theta_ceil", "error_clip", "m_norm_max")
_DECODE_RULE = {"hebbian": 0, "delta": 1, "titans": 1, "dgd": 2}


def _decode_plan(params, cfg, active, context, kv_cache, ws, tensors):
    """The argument block of the one-call step, or None for a model that it does not cover (MLP memories, SwiGLU, other
    head sizes): those take the step below, operation by operation."""
    d, nh, hd, v, k = cfg.d_model, cfg.num_heads, cfg.head_dim, cfg.vocab_size, cfg.k
    if (hd not in (32, 64, 128) or nh * hd != d or d > 4096 or not 1 <= k <= 8 or kv_cache._scratch_k.numel() < d
            or kv_cache.d != d):
        return None
    for i, t in enumerate(ws.written()):
        if (t.dtype != (torch.bfloat16 if i in (1, 2) else torch.float32) or not t.is_cuda or not t.is_contiguous()
                or tuple(t.shape) != (1, v if i == 7 else d) or t.data_ptr() & 15):
            return None
    host = ws.logits_host
    if host.dtype != torch.float32 or host.is_cuda or not host.is_pinned() or not host.is_contiguous() or host.shape != (v,):
        return None
    square, vectors = [params.w_q, params.w_k, params.w_v, params.w_o], []
    rules, bounds = [], []
    for lv in range(k):
        lc, lp, mem = cfg.levels[lv], params.levels[lv], context.memory[lv]
        rule = _DECODE_RULE.get(lc.memory_rule)
        if rule is None or lc.memory_layers != 1 or (lc.num_heads, lc.head_dim) != (nh, hd):
            return None
        if mem.shape != (nh, hd * hd) and (active[lv] or mem[:nh].numel() != nh * hd * hd):
            return None
        rules.append(rule if active[lv] else -1)
        bounds += (lc.alpha_floor, lc.alpha_ceil, lc.theta_floor, lc.theta_ceil, lc.error_clip, lc.m_norm_max)
        square += (lp.w_k, lp.w_v, lp.w_q)
        vectors += (lp.w_alpha, lp.w_theta)
    if (any(t.shape != (d, d) for t in square) or any(t.numel() != 2 * d for t in vectors)
            or params.w_unembed.shape != (d, v) or params.w_embed.shape != (v, d)):
        return None
    # contiguous on the device, read in 16-byte pieces (all but the scalar biases); floats except for the two caches
    for i, t in enumerate(tensors):
        cache = i in (6, 7)
        if (t.dtype != (torch.bfloat16 if cache else torch.float32) or not t.is_cuda or not t.is_contiguous() or t.numel() == 0
                or (t.numel() > 1 and t.data_ptr() & 15) or (cache and t.numel() < kv_cache.max_len * d)):
            return None
    if len({m.data_ptr() for m in context.memory[:k]}) < k:   # levels that share a memory take it in turn
        return None
    work = ws.work_for(lib.decode_work_floats_rocm(d, nh, k, min(cfg.window_size, kv_cache.max_len), cfg.n_persistent))
    ptrs = [t.data_ptr() for t in tensors]
    weights = ptrs[1:6]
    level_args = ((ctypes.c_void_p * (8 * k))(*ptrs[8:]), (ctypes.c_int * k)(*rules), (ctypes.c_float * (6 * k))(*bounds))
    written = [t.data_ptr() for t in ws.written()]
    tail = (kv_cache.k_cache_bf16.data_ptr(), kv_cache.v_cache_bf16.data_ptr(), work.data_ptr(), (ctypes.c_void_p * 7)(*written[:7]),
            written[7], ws.logits_host.data_ptr())
    return ptrs[0], weights, level_args, tail


def _decode_in_one_call(params, cfg, token_id, pulse, context, kv_cache, ws):
    """The whole step as one library call -> logits, or None (see _decode_plan).  Checking some forty tensors and level
    options costs as much as the step's kernels, so the workspace keeps the argument blocks together with everything they
    were made from (addresses, sizes, strides, types, options, pulse) and makes one again when any of it has changed."""
    k = cfg.k
    if not _keys_fit(cfg, kv_cache.len):
        return None
    levels, lcfgs = params.levels, cfg.levels
    tensors = [params.w_embed, params.w_q, params.w_k, params.w_v, params.w_o, params.w_unembed, kv_cache.k_cache_bf16,
               kv_cache.v_cache_bf16]
    active = tuple(map(bool, pulse.active_levels[:k]))
    options = [cfg.d_model, cfg.num_heads, cfg.head_dim, cfg.vocab_size, cfg.window_size, cfg.n_persistent, kv_cache.d,
               kv_cache.max_len]
    for lv in range(k):
        lp = levels[lv]
        if not hasattr(lp, "w_alpha"):
            return None
        tensors += _LEVEL_TENSORS(lp)
        tensors.append(context.memory[lv])
        options += _LEVEL_OPTIONS(lcfgs[lv])
    # a tensor can be transposed or resized where it stands: sizes and strides are read anew as well as the address
    key = (options, ffi.tensor_key([*tensors, *ws.written(), kv_cache._scratch_k, ws.logits_host]))
    made_for, plan = ws.plans.get(active, (None, None))
    if made_for != key:
        plan = _decode_plan(params, cfg, active, context, kv_cache, ws, tensors)
        if len(ws.plans) >= 16:
            ws.plans.clear()
        ws.plans[active] = (key, plan)
    if plan is None:
        return None
    rows, weights, level_args, tail = plan
    rc = lib.decode_token_rocm(rows + 4 * cfg.d_model * token_id, *weights, *level_args, k, cfg.d_model,
                               cfg.num_heads, cfg.vocab_size, cfg.window_size, cfg.n_persistent, kv_cache.len, *tail)
    if rc:
        raise RuntimeError(f"decode_token_rocm failed ({rc})")
    kv_cache.len += 1
    return ws.logits_host.numpy().copy()


def _memory_read_only(lp, embedded, memory, n, nh, hd):
    """gpu_memory_read_only (:2906-2950): y = M_h q per head with the raw projection q and the memories of the
    first batch slot."""
    q = (embedded @ lp.w_q.t()).contiguous()
    y = _new(n, nh * hd)
    D.call("memory_read_only_f32_rocm", q, memory[:nh].contiguous(), y, n, nh, hd)
    return y


def frozen_level_output(lcfg, lp, embedded, memory, n, nh, hd, level):
    """What a frozen level contributes (gpu_forward.rs:1008-1024, 3255-3265, 3449-3459): the read y = M_h q for a
    matrix memory; zeros for MONETA / YAAD, whose context memory is the flat [W1 | W2] block that the matrix read
    cannot interpret (frozen_mlp_fallback, :45-57); an error for the two-layer Titans memory
    (panic_if_frozen_titans_mlp, :32-39)."""
    if lcfg.is_mlp_mem:
        raise RuntimeError(f"Frozen TitansLMM MLP level unsupported (level {level}): read-only MLP kernel not implemented")
    if lcfg.memory_rule in ("moneta", "yaad"):
        return _zeros(n, nh * hd)
    return _memory_read_only(lp, embedded, memory, n, nh, hd)


def _levels(params, cfg, embedded, pulse, context, s):
    ys = []
    for level in range(cfg.k):
        if pulse.active_levels[level]:
            y, _cache = gpu_memory_forward(params.levels[level], cfg.levels[level], embedded, context.memory[level], s,
                                           cfg.d_model, 1)
        else:
            y = frozen_level_output(cfg.levels[level], params.levels[level], embedded, context.memory[level], s,
                                    cfg.num_heads, cfg.head_dim, level)
        ys.append(y)
    return ys


def _combine_gate(ys, attn_out, y_combined, gate, gated, n):
    """Sum of the levels (times 1/sqrt(k) for k > 2), sigmoid gate on the attention output (:3275-3293)."""
    ptrs = (ctypes.c_void_p * len(ys))(*[y.data_ptr() for y in ys])
    lib.cms_combine_gate_rocm(ptrs, len(ys), attn_out.data_ptr(), y_combined.data_ptr(), gate.data_ptr(),
                              gated.data_ptr(), n)


def _prefill_in_batch(params, cfg, input_ids, pulse, context):
    """A prompt leaves three things behind: K and V of every token, the levels' memories after the last token, and the
    logits of the last position.  So only k, v and the gates are formed for every token (one group of products, one pass
    of glue over all active levels), the memories go straight to their final states, and the last position is one decode
    step that reads them: attention, combine, gate, output projection and unembedding of one token.  Exact Delta, Titans
    and DGD levels without clip or bound and frozen matrix levels; None: anything else takes the step below."""
    s, d, nh, hd, v, k = cfg.seq_len, cfg.d_model, cfg.num_heads, cfg.head_dim, cfg.vocab_size, cfg.k
    if hd not in (32, 64, 128) or nh * hd != d or d > 1024 or not 1 <= k <= 8 or s < 1 or params.w_embed.shape != (v, d):
        return None
    if not _keys_fit(cfg, s - 1):
        return None
    active = [lv for lv in range(k) if pulse.active_levels[lv]]
    keys = {group_key(cfg.levels[lv], params.levels[lv], d, 1) for lv in active}
    if len(keys) > 1 or None in keys:
        return None
    for lv in range(k):
        lc, lp, mem = cfg.levels[lv], params.levels[lv], context.memory[lv]
        if (_DECODE_RULE.get(lc.memory_rule) is None or lc.memory_layers != 1 or (lc.num_heads, lc.head_dim) != (nh, hd)
                or not _plain(mem, nh, hd * hd)):
            return None
        if pulse.active_levels[lv]:   # its parameters have a key
            if lc.error_clip > 0 or 0 < lc.m_norm_max < 1e30 or lc.proxy:
                return None
        elif not all(_plain(t, d, d) for t in (lp.w_k, lp.w_v, lp.w_q)):
            return None
    if len({m.data_ptr() for m in context.memory[:k]}) < k:
        return None
    if (not _plain(params.w_embed, v, d) or not _plain(params.w_unembed, d, v)
            or not all(_plain(w, d, d) for w in (params.w_q, params.w_k, params.w_v, params.w_o))):
        return None
    pinned = torch.empty(s, dtype=torch.int32, pin_memory=True)
    ids = pinned.numpy()
    ids[:] = host_ids(input_ids[:s])
    last = int(ids[s - 1])
    if ids.min() < 0 or ids.max() >= v:
        return None
    embedded, dev_ids = _new(s, d), pinned.cuda(non_blocking=True)   # by name: alive until the call has launched
    lib.embedding_gather_cuda(params.w_embed.data_ptr(), dev_ids.data_ptr(), embedded.data_ptr(), s, d)
    kv_cache = GpuKVCache(s + cfg.decode_tokens, d, s)
    L = len(active)
    mem = list(_new(max(2 * L, 1), s, d).unbind(0))[:2 * L]
    weights = [w for lv in active for w in (params.levels[lv].w_k, params.levels[lv].w_v)] + [params.w_k, params.w_v]
    linear_group(0, [embedded] * (2 * L + 2), weights, mem + [kv_cache.k_cache_bf16, kv_cache.v_cache_bf16], s, d, d, 3 << (2 * L))
    kv_cache.len = s
    if L:
        cfgs, lps = [cfg.levels[lv] for lv in active], [params.levels[lv] for lv in active]
        titans = cfgs[0].memory_rule == "titans"
        heads, gates = _new(2, L * nh, s, hd), _new(3 if titans else 2, L * nh, s)
        rows = list(_new(4 * L, s).unbind(0))
        h0, g0 = heads.data_ptr(), gates.data_ptr()
        hs, gs = 4 * L * nh * s * hd, 4 * L * nh * s
        lib.level_group_inputs_f32_rocm(
            _ptrs([t for i, lp in enumerate(lps) for t in (
                mem[2 * i], mem[2 * i + 1], mem[2 * i], *_gate_params(lp, titans), rows[4 * i], rows[4 * i], rows[4 * i + 1],
                rows[4 * i + 2], rows[4 * i + 3])]),
            (ctypes.c_float * (4 * L))(*[x for c in cfgs for x in (c.alpha_floor, c.alpha_ceil, c.theta_floor, c.theta_ceil)]), L,
            h0, h0 + hs, None, g0, g0 + gs, g0 + 2 * gs if titans else None, 1, s, nh, hd, 1e-8)
        contexts = [context.memory[lv] for lv in active]
        states = contexts[0]
        if L > 1:
            states = _new(L * nh, hd * hd)
            lib.level_group_states_gather_rocm(_ptrs(contexts), L, states.data_ptr(), nh, hd * hd)
        if titans:
            lib.titans_final_states_f32_rocm(h0, h0 + hs, g0, g0 + gs, g0 + 2 * gs, states.data_ptr(), None, states.data_ptr(), s, hd,
                                             L * nh)
        else:
            lib.delta_final_states_f32_rocm(h0, h0 + hs, g0, g0 + gs, states.data_ptr(), states.data_ptr(), s, hd, L * nh)
        if L > 1:
            lib.level_group_states_final_rocm(states.data_ptr(), hd * hd, _ptrs(contexts), (ctypes.c_float * L)(*[F32_MAX] * L), L,
                                              nh, hd * hd)
    # the last position as a decode step at a cache row that holds its K and V already
    level_ptrs = [t.data_ptr() for lv in range(k) for lp in (params.levels[lv],) for t in (
        lp.w_k, lp.w_v, lp.w_q, lp.w_alpha, lp.b_alpha, lp.w_theta, lp.b_theta, context.memory[lv])]
    work = _new(lib.decode_work_floats_rocm(d, nh, k, min(cfg.window_size, s), cfg.n_persistent) + 7 * d + v)
    w0 = work.data_ptr()
    row, step = w0 + 4 * (work.numel() - 7 * d - v) // 16 * 16, 4 * d
    outputs = (ctypes.c_void_p * 7)(*[row + i * step for i in range(7)])
    logits = torch.empty(v, dtype=torch.float32, pin_memory=True)
    rc = lib.decode_token_rocm(
        params.w_embed.data_ptr() + 4 * d * last, params.w_q.data_ptr(), params.w_k.data_ptr(), params.w_v.data_ptr(),
        params.w_o.data_ptr(), params.w_unembed.data_ptr(), (ctypes.c_void_p * (8 * k))(*level_ptrs),
        (ctypes.c_int * k)(*[3 if pulse.active_levels[lv] else -1 for lv in range(k)]), (ctypes.c_float * (6 * k))(), k, d, nh, v,
        cfg.window_size, cfg.n_persistent, s - 1, kv_cache.k_cache_bf16.data_ptr(), kv_cache.v_cache_bf16.data_ptr(), w0, outputs,
        row + 7 * step, logits.data_ptr())
    if rc:
        raise RuntimeError(f"decode_token_rocm failed ({rc})")
    return logits.numpy().copy(), kv_cache


def gpu_prefill_forward(params: GpuMAGParams, cfg: ServeConfig, input_ids, pulse: Pulse, context: ContextState):
    """-> (logits of the last prompt position [vocab] on the host, GpuKVCache holding the prompt)."""
    s, d, nh, hd = cfg.seq_len, cfg.d_model, cfg.num_heads, cfg.head_dim
    assert d == nh * hd
    assert not cfg.residual, "gpu_prefill_forward: residual=true is not served by the cached-generation path"
    assert len(input_ids) >= s
    done = _prefill_in_batch(params, cfg, input_ids, pulse, context)
    if done is not None:
        return done
    ids = torch.tensor([int(t) for t in input_ids[:s]], dtype=torch.int32).cuda()
    embedded = _new(s, d)
    D.call("embedding_gather_cuda", params.w_embed, ids, embedded, s, d)
    q_f32, k_f32, v_f32 = (embedded @ w.t() for w in (params.w_q, params.w_k, params.w_v))
    kv_cache = GpuKVCache(s + cfg.decode_tokens, d, s)
    kv_cache.append_f32(k_f32, v_f32, s)
    q_bf16 = _new(s, d, dtype=torch.bfloat16)
    D.call("f32_to_bf16_cuda", q_f32, q_bf16, s * d)
    attn_out_bf16 = _new(s, d, dtype=torch.bfloat16)
    attn_weights = _new(nh, s, cfg.n_persistent + cfg.window_size, dtype=torch.bfloat16)
    k_bf16 = kv_cache.k_cache_bf16[:s].contiguous()
    v_bf16 = kv_cache.v_cache_bf16[:s].contiguous()
    D.call("swa_forward_f32_cuda", q_bf16, k_bf16, v_bf16, attn_out_bf16, attn_weights, s, nh, hd, cfg.window_size,
           1, cfg.n_persistent)
    attn_out = _new(s, d)
    D.call("bf16_to_f32_cuda", attn_out_bf16, attn_out, s * d)
    ys = _levels(params, cfg, embedded, pulse, context, s)
    y_combined, gate, gated = _new(s, d), _new(s, d), _new(s, d)
    _combine_gate(ys, attn_out, y_combined, gate, gated, s * d)
    projected = gated @ params.w_o.t()
    logits = projected[s - 1:s] @ params.w_unembed
    return logits[0].cpu().numpy(), kv_cache


def gpu_single_token_forward(params: GpuMAGParams, cfg: ServeConfig, token_id, pulse: Pulse, context: ContextState,
                             kv_cache: GpuKVCache, ws: DecodeWorkspace):
    """One decode step -> logits [vocab] on the host."""
    d, v, nh, hd = cfg.d_model, cfg.vocab_size, cfg.num_heads, cfg.head_dim
    assert not cfg.residual, "gpu_single_token_forward: residual=true is not served by the cached-generation path"
    if not 0 <= token_id < v:
        raise ValueError(f"token_id {token_id} >= vocab_size {v}")
    token_id = int(token_id)   # a numpy whole number or a 0-d tensor, as argmax of the logits gives
    if kv_cache.len == 0:
        raise RuntimeError("KV cache must be populated via prefill first")
    if kv_cache.len >= kv_cache.max_len:
        raise OverflowError(f"KV cache full: {kv_cache.len} >= {kv_cache.max_len}")
    logits = _decode_in_one_call(params, cfg, token_id, pulse, context, kv_cache, ws)
    if logits is not None:
        return logits
    ws.d_input.copy_(torch.tensor([token_id], dtype=torch.int32))
    D.call("embedding_gather_cuda", params.w_embed, ws.d_input, ws.embedded, 1, d)
    q_f32, k_f32, v_f32 = (ws.embedded @ w.t() for w in (params.w_q, params.w_k, params.w_v))
    kv_cache.append_f32(k_f32, v_f32, 1)
    D.call("f32_to_bf16_cuda", q_f32, ws.q_bf16, d)
    D.call("swa_single_token_cuda", ws.q_bf16, kv_cache.k_cache_bf16, kv_cache.v_cache_bf16, ws.attn_out_bf16,
           kv_cache.len, nh, hd, cfg.window_size, cfg.n_persistent)
    D.call("bf16_to_f32_cuda", ws.attn_out_bf16, ws.attn_out, d)
    ys = _levels(params, cfg, ws.embedded, pulse, context, 1)
    _combine_gate(ys, ws.attn_out, ws.y_combined, ws.gate, ws.gated_out, d)
    projected = ws.gated_out @ params.w_o.t()
    torch.mm(projected, params.w_unembed, out=ws.logits_gpu)
    return ws.logits_gpu[0].cpu().numpy()
