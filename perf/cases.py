"""Cases that stand for the work a user of this library has it do on one GPU, each through the public entry points.

Families (the `kind` of a case) and their real use:
  decode     cached generation, one token after the other: a reply of a few tokens to a prompt that is in the cache
  prefill    cached generation: the forward pass over a prompt that fills the cache
  train      one training step of the whole model from token ids (forward, backward, SGD), levels with the full state
             trajectory, which is the reference's default, or as frozen-M0 chunkwise levels under its m_norm_max
  layer      one training step of the tuned layer (levels, sliding-window attention, gate, frequency-aware AdamW)
  chunk_bf16 the frozen-M0 chunkwise rule on bf16 tokens, forward and backward
  chunk_f32  the same on float tokens through the reference-named symbols, with the m_norm_max its configurations ship
  exact      the exact per-token rule with state checkpoints, forward and backward
  hope       the self-referential memory, forward and backward
  attn       sliding-window attention with the weights stored (the reference's contract), forward and backward
"""
import math

import torch

from nl_hecate_amd import cms_model as CM
from nl_hecate_amd import dispatch as D
from nl_hecate_amd import selfref as SR
from nl_hecate_amd import serving as SV
from nl_hecate_amd.cms import Conductor, ContextState
from nl_hecate_amd.mag_layer import MagLayer, MagTrainer, MemoryLevelParams
from nl_hecate_amd.memory_level import LevelConfig, checkpoint_count

F32_MAX = 3.4028234663852886e38
PERIODS = [1, 8, 64, 512]   # chunk sizes of the four levels


def listed():
    return [
        # the smallest calls: sixteen tokens of a reply, each waiting for the one before; launches and latency count
        dict(name="decode_reply", kind="decode", rule="titans", heads=8, head_dim=64, levels=4, window=512, vocab=32000,
             prompt=640, tokens=16),
        # an ordinary prompt, its length no multiple of anything
        dict(name="prefill_prompt", kind="prefill", rule="titans", heads=8, head_dim=64, levels=4, window=512, vocab=32000,
             prompt=1000),
        # the model size that the reference quotes its training rate for (d = 512, four levels, 512 tokens)
        dict(name="train_trajectory", kind="train", rule="titans", heads=8, head_dim=64, levels=4, window=512, vocab=32000,
             batch=1, seq=512, proxy=False),
        # levels by the frozen-M0 chunkwise rule with a norm bound, head size 32 as in the reference's 1024-wide model
        dict(name="train_proxy_hd32", kind="train", rule="delta", heads=16, head_dim=32, levels=2, window=256, vocab=8000,
             batch=2, seq=1000, proxy=True),
        # a fine-tuning step: short sequences, narrow model
        dict(name="layer_small", kind="layer", heads=4, levels=2, window=256, batch=1, seq=500),
        # the full layer at its training size: the largest step
        dict(name="layer_large", kind="layer", heads=8, levels=4, window=512, batch=8, seq=4096),
        # the rule alone at its training size: 16 sequences of 8 heads
        dict(name="chunk_bf16_large", kind="chunk_bf16", rule="titans", chains=128, seq=4096, chunk=64),
        # an ordinary batch, ragged length, through the symbols that a caller of the reference has
        dict(name="chunk_f32_bounded", kind="chunk_f32", rule="titans", chains=32, seq=1500, chunk=64),
        # the exact rule at its training size: 8 sequences of 8 heads
        dict(name="exact_large", kind="exact", rule="titans", head_dim=64, chains=64, seq=2048, interval=64),
        # the exact rule without momentum, few short chains of head size 32
        dict(name="exact_delta_hd32", kind="exact", rule="delta", head_dim=32, chains=16, seq=777, interval=64),
        # the self-referential memory at its training size
        dict(name="hope_large", kind="hope", chains=64, seq=2048, chunk=64),
        # attention of the layer through the reference's contract
        dict(name="attn_large", kind="attn", heads=8, head_dim=64, batch=8, seq=4096, window=512),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, even over the logarithm, odd ones among them."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("decode", "prefill", "train", "layer", "chunk_bf16", "chunk_f32", "exact", "hope", "attn"))
    rule = rng.choice(("titans", "titans", "delta"))
    head_dim = rng.choice((64, 64, 32))
    heads = rng.choice((4, 8, 16))
    model = dict(rule=rule, heads=heads, head_dim=head_dim, levels=rng.randint(1, 4), window=rng.choice((128, 256, 512)),
                 vocab=_log(rng, 1000, 32000))
    if kind == "decode":
        return dict(kind=kind, **model, prompt=_log(rng, 8, 2000), tokens=rng.randint(1, 16))
    if kind == "prefill":
        return dict(kind=kind, **model, prompt=_log(rng, 16, 1000))
    if kind == "train":
        proxy = rng.random() < 0.5
        batch = rng.randint(1, 2) if heads < 16 else 1
        return dict(kind=kind, **model, batch=batch, seq=_log(rng, 64, 1000 if proxy else 512) // batch, proxy=proxy)
    if kind == "layer":
        seq = _log(rng, 128, 4096)
        return dict(kind=kind, heads=rng.choice((4, 8)), levels=rng.randint(1, 4), window=rng.choice((128, 256, 512)),
                    batch=rng.randint(1, 8), seq=seq)
    if kind == "chunk_bf16":
        return dict(kind=kind, rule=rule, chains=_log(rng, 8, 128), seq=_log(rng, 64, 4096), chunk=rng.choice((32, 64, 64)))
    if kind == "chunk_f32":
        return dict(kind=kind, rule=rule, chains=_log(rng, 8, 64), seq=_log(rng, 64, 2048), chunk=rng.choice((32, 64, 64)))
    if kind == "exact":
        return dict(kind=kind, rule=rule, head_dim=head_dim, chains=_log(rng, 4, 64), seq=_log(rng, 64, 2048),
                    interval=rng.choice((32, 64, 64)))
    if kind == "hope":
        return dict(kind=kind, chains=_log(rng, 4, 64), seq=_log(rng, 100, 2048), chunk=rng.choice((32, 64)))
    seq = _log(rng, 128, 4096)
    return dict(kind=kind, heads=8 if head_dim == 64 else 16, head_dim=head_dim, batch=rng.randint(1, 8 if head_dim == 64 else 5),
                seq=seq, window=rng.choice((128, 256, 512)))


# ── what a user's program has in hand ────────────────────────────────────────────────────────────────────────────

class _Rand:
    """Seeded device tensors of the distributions that the paths meet."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed & 0x7fffffff)

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, generator=self.g, device="cuda") * std

    def xavier(self, rows, cols):
        return (torch.rand(rows, cols, generator=self.g, device="cuda") * 2 - 1) * math.sqrt(6.0 / (rows + cols))

    def unit(self, *shape):
        x = self.normal(*shape)
        return x / x.norm(dim=-1, keepdim=True)

    def gate(self, *shape):
        return torch.sigmoid(self.normal(*shape))

    def ids(self, n, vocab):
        return torch.randint(0, vocab, (n,), generator=self.g, device="cuda").tolist()


def _model_params(r, c):
    """Weights of the whole model and each level's carried memory, one matrix per (batch element, head)."""
    d, v, hd = c["heads"] * c["head_dim"], c["vocab"], c["head_dim"]
    one = lambda x: torch.full((1,), x, device="cuda")
    vec = lambda: (torch.rand(2 * d, generator=r.g, device="cuda") * 2 - 1) * 0.05
    levels = [MemoryLevelParams(r.xavier(d, d), r.xavier(d, d), r.xavier(d, d), vec(), one(-2.0), vec(), one(-3.0), vec(),
                                one(2.0)) for _ in range(c["levels"])]
    params = SV.GpuMAGParams(r.normal(v, d), r.xavier(d, d), r.xavier(d, d), r.xavier(d, d), r.xavier(d, d), r.xavier(d, v),
                             levels)
    context = ContextState([r.normal(c.get("batch", 1) * c["heads"], hd * hd, std=0.05) for _ in range(c["levels"])])
    return params, context


def _level_configs(c):
    more = dict(proxy=True, chunk_size=64, m_norm_max=100.0) if c.get("proxy") else {}
    return [LevelConfig(c["rule"], c["heads"], c["head_dim"], **more) for _ in range(c["levels"])]


def prepare(case, seed):
    c, r = dict(case), _Rand(seed)
    kind = c["kind"]
    st = dict(case=c)
    if kind in ("decode", "prefill"):
        d, hd = c["heads"] * c["head_dim"], c["head_dim"]
        st["params"], st["context"] = _model_params(r, c)
        st["conductor"] = Conductor(c["levels"], PERIODS[:c["levels"]])
        st["cfg"] = SV.ServeConfig(d, c["vocab"], c["heads"], hd, c["window"], c["prompt"], _level_configs(c),
                                   decode_tokens=64)
        st["prompt"] = r.ids(c["prompt"], c["vocab"])
        if kind == "decode":
            st["kv"] = SV.GpuKVCache(c["prompt"] + 64, d, c["prompt"])
            st["kv"].append_f32(r.normal(c["prompt"], d), r.normal(c["prompt"], d), c["prompt"])
            st["ws"] = SV.DecodeWorkspace(d, c["vocab"])
            st["reply"] = r.ids(c["tokens"], c["vocab"])
            st["conductor"].set_seq_len(1)
        else:
            st["conductor"].set_seq_len(c["prompt"])
        return st
    if kind == "train":
        d = c["heads"] * c["head_dim"]
        st["params"], st["context"] = _model_params(r, c)
        st["conductor"] = Conductor(c["levels"], PERIODS[:c["levels"]])
        st["conductor"].set_seq_len(c["seq"])
        st["cfg"] = CM.ModelConfig(d, c["vocab"], c["heads"], c["head_dim"], c["window"], c["seq"], _level_configs(c))
        st["ids"] = r.ids(c["batch"] * c["seq"], c["vocab"])
        st["targets"] = r.ids(c["batch"] * c["seq"], c["vocab"])
        return st
    if kind == "layer":
        d = 64 * c["heads"]
        layer = MagLayer(d, c["heads"], c["levels"], c["window"], PERIODS[:c["levels"]], rule="chunkwise", chunk=64,
                         seed=seed & 0xffff, precision="bf16")
        st["trainer"] = MagTrainer(layer, lr=3e-5, beta1=0.9, beta2=0.95, weight_decay=0.1)
        st["x"] = r.normal(c["batch"], c["seq"], d, std=d ** -0.5)
        st["d_out"] = r.normal(c["batch"], c["seq"], d)
        return st
    f32 = lambda *shape: torch.zeros(*shape, device="cuda")
    if kind == "attn":
        b, s, h, hd, w = c["batch"], c["seq"], c["heads"], c["head_dim"], c["window"]
        st["q"], st["k"], st["v"] = (r.normal(b, s, h * hd).to(torch.bfloat16) for _ in range(3))
        st["d_out"] = r.normal(b, s, h * hd)
        st["out"] = torch.zeros(b, s, h * hd, dtype=torch.bfloat16, device="cuda")
        st["weights"] = torch.zeros(b, h, s, w, dtype=torch.bfloat16, device="cuda")
        st["d_q"], st["d_k"], st["d_v"] = (f32(b, s, h * hd) for _ in range(3))
        return st
    B, s = c["chains"], c["seq"]
    if kind == "hope":
        d = 64
        # memories that are all live, with a decay gate that starts low, so that they carry data over many tokens
        u = torch.full((d,), d ** -0.5, device="cuda")
        lim = math.sqrt(6.0 / (2 * d))
        mems = (torch.rand(B, 6, d, d, generator=r.g, device="cuda") * 2 - 1) * lim
        mems[:, 4] -= 13.0 * u
        mems[:, 3] -= 6.0 * u
        st["mems"] = mems
        st["x"] = r.normal(B, s, d, std=(8 * d) ** -0.5) + 0.5 * u
        st["d_y"] = r.normal(B, s, d)
        return st
    d = c.get("head_dim", 64)
    tok = (lambda x: x.to(torch.bfloat16)) if kind == "chunk_bf16" else (lambda x: x)
    st["k"], st["v"], st["q"] = tok(r.unit(B, s, d)), tok(r.normal(B, s, d)), tok(r.unit(B, s, d))
    st["gates"] = [r.gate(B, s) for _ in range(3 if c["rule"] == "titans" else 2)]
    st["d_y"] = r.normal(B, s, d)
    n_mats = 2 if c["rule"] == "titans" else 1
    slots = checkpoint_count(s, c["interval"]) if kind == "exact" else -(-s // c["chunk"]) + 1
    st["initial"] = [r.normal(B, d, d, std=0.1)] + [f32(B, d, d)] * (n_mats - 1)
    st["states"] = [f32(B, slots, d, d) for _ in range(n_mats)]
    st["y"] = f32(B, s, d)
    st["grads"] = [f32(B, s, d) for _ in range(3)] + [f32(B, s) for _ in st["gates"]]
    st["d_initial"] = [f32(d, d) for _ in range(n_mats)]
    return st


# ── one pass ─────────────────────────────────────────────────────────────────────────────────────────────────────

def run(st):
    c = st["case"]
    return _RUN[c["kind"]](st, c)


def _decode(st, c):
    kv, cond = st["kv"], st["conductor"]
    kv.len = c["prompt"]   # the reply is generated again behind the same prompt
    logits = []
    for t in st["reply"]:
        logits.append(SV.gpu_single_token_forward(st["params"], st["cfg"], t, cond.pulse(), st["context"], kv, st["ws"]))
        cond.advance()
    return {"logits": logits, "memory": st["context"].memory, "k_cache": kv.k_cache_bf16, "v_cache": kv.v_cache_bf16}


def _prefill(st, c):
    logits, kv = SV.gpu_prefill_forward(st["params"], st["cfg"], st["prompt"], st["conductor"].pulse(), st["context"])
    return {"logits": logits, "memory": st["context"].memory, "k_cache": kv.k_cache_bf16, "v_cache": kv.v_cache_bf16}


def _train(st, c):
    p, cfg = st["params"], st["cfg"]
    loss, cache = CM.gpu_cms_forward(p, cfg, st["ids"], st["targets"], st["conductor"].pulse(), st["context"])
    g = CM.gpu_cms_backward(p, cfg, cache)
    CM.gpu_weight_update(p, g, 1e-2)
    st["conductor"].advance()
    level = lambda x: [x.d_w_k_mem, x.d_w_v_mem, x.d_w_q_mem, x.d_w_alpha, x.d_b_alpha, x.d_w_theta, x.d_b_theta] + (
        [x.d_w_eta, x.d_b_eta] if c["rule"] == "titans" else [])
    return {"loss": loss, "grads": [g.d_w_embed, g.d_w_q, g.d_w_k, g.d_w_v, g.d_w_o, g.d_w_unembed],
            "level_grads": [level(x) for x in g.levels], "memory": st["context"].memory,
            "params": [p.w_embed, p.w_q, p.w_k, p.w_v, p.w_o, p.w_unembed]}


def _layer(st, c):
    tr = st["trainer"]
    out = tr.step_graphed(st["x"], st["d_out"])
    return {"out": out, "grads": tr.grads.flat, "params": tr.layer.p.tensors(), "m": tr.layer.m_state, "s": tr.layer.s_state}


def _rule(st, forward, backward, sizes, tail):
    """Forward and backward of a rule; the gradients of the initial states are sums that the caller starts at zero."""
    for t in st["d_initial"]:
        t.zero_()
    kvq = (st["k"], st["v"], st["q"])
    D.call(forward, *kvq, *st["gates"], *st["initial"], *st["states"], st["y"], *sizes, *tail)
    D.call(backward, *kvq, *st["gates"], *st["states"], st["d_y"], *st["grads"], *st["d_initial"], *sizes, *tail)
    return {"y": st["y"], "states": st["states"], "grads": st["grads"], "d_initial": st["d_initial"]}


def _chunk_bf16(st, c):
    return _rule(st, f"{c['rule']}_chunkwise_forward_bf16_rocm", f"{c['rule']}_chunkwise_backward_bf16_rocm",
                 (c["seq"], 64, c["chains"], c["chunk"]), ())


def _chunk_f32(st, c):
    return _rule(st, f"{c['rule']}_chunkwise_forward_f32_cuda", f"{c['rule']}_chunkwise_backward_f32_cuda",
                 (c["seq"], 64, c["chains"], c["chunk"]), (0.0, 100.0))


def _exact(st, c):
    return _rule(st, f"{c['rule']}_forward_ckpt_batched_f32_rocm", f"{c['rule']}_backward_ckpt_f32_rocm",
                 (c["seq"], c["head_dim"], c["chains"], c["interval"]), (0.0, F32_MAX))


def _hope(st, c):
    mems = st["mems"].clone()   # the step updates them in place
    y, cache = SR.chunkwise_self_ref_step(mems, st["x"], c["chunk"], True)
    d_x, d_mems = SR.chunkwise_self_ref_step_backward(cache, st["d_y"])
    return {"y": y, "mems": mems, "d_x": d_x, "d_mems": d_mems}


def _attn(st, c):
    sizes = (c["seq"], c["heads"], c["head_dim"], c["window"], c["batch"], 0)
    D.call("swa_forward_f32_cuda", st["q"], st["k"], st["v"], st["out"], st["weights"], *sizes)
    st["d_k"].zero_()
    st["d_v"].zero_()
    D.call("swa_backward_f32_cuda", st["q"], st["k"], st["v"], st["weights"], st["d_out"], st["d_q"], st["d_k"], st["d_v"],
           *sizes)
    return {"out": st["out"], "weights": st["weights"], "d_q": st["d_q"], "d_k": st["d_k"], "d_v": st["d_v"]}


_RUN = dict(decode=_decode, prefill=_prefill, train=_train, layer=_layer, chunk_bf16=_chunk_bf16, chunk_f32=_chunk_f32,
            exact=_exact, hope=_hope, attn=_attn)


# ── what a pass cannot do without ────────────────────────────────────────────────────────────────────────────────

def _rule_work(tokens, d, mats, state_slots, token_bytes, flops_per_token):
    """tokens = chains * length.  Forward: k, v, q, gates in, y out; backward: those and d_y in, three gradients and the
    gates' out; the kept states written once and read once."""
    gates = 4 * (mats + 1)
    fwd = 3 * token_bytes * d + gates + 4 * d
    bwd = 3 * token_bytes * d + gates + 4 * d + 12 * d + gates
    return tokens * (fwd + bwd) + 2 * mats * state_slots * 4 * d * d, tokens * flops_per_token


def _pairs(s, w):
    """Query-key pairs of one head and sequence under a causal window."""
    w = min(w, s)
    return s * w - w * (w - 1) // 2


def work(case):
    c = case
    kind = c["kind"]
    if kind in ("decode", "prefill", "train"):
        d, hd, v, k = c["heads"] * c["head_dim"], c["head_dim"], c["vocab"], c["levels"]
        weights = 4 * ((4 + 3 * k) * d * d + 6 * d * k)
        mem = 4 * k * c.get("batch", 1) * d * hd
        rule = (9 if c["rule"] == "titans" else 6) * d * hd   # forward of one token over all heads of a level
        if kind == "decode":
            n, L = c["tokens"], min(c["window"], c["prompt"] + c["tokens"])
            # one token at a time: every weight once per token; only the first level is sure to be active
            per = 4 * (4 + 3 + (k - 1)) * d * d + 4 * d * v + 4 * L * d + 2 * mem + 4 * v
            return {"bytes": n * per, "flops": n * (2 * (4 + 3 + (k - 1)) * d * d + 2 * d * v + 4 * L * d + rule)}
        if kind == "prefill":
            n = c["prompt"]
            return {"bytes": weights + 4 * d * v + 2 * mem + 4 * n * d + 4 * n * d,
                    "flops": 2 * n * (4 + 3 * k) * d * d + 2 * d * v + 4 * _pairs(n, c["window"]) * d + n * k * rule}
        n = c["batch"] * c["seq"]
        # forward, backward and update: weights read and written, embedding rows, the loss over the vocabulary
        return {"bytes": 2 * (weights + 8 * d * v) + 4 * mem,
                "flops": 6 * n * (4 + 3 * k) * d * d + 6 * n * d * v + 14 * c["batch"] * _pairs(c["seq"], c["window"]) * d
                + n * k * rule * 3}
    if kind == "layer":
        n, d, k = c["batch"] * c["seq"], 64 * c["heads"], c["levels"]
        by, fl = _rule_work(n * c["heads"] * k, 64, 2, c["batch"] * c["heads"] * k * (-(-c["seq"] // 64) + 1), 2, 200704)
        params = (4 + 3 * k) * d * d + 6 * d * k
        # x, d_out, out, d_x, the attention's q, k, v and gradients in bf16, parameters with their optimizer state
        by += n * d * (16 + 16) + 28 * params
        fl += 6 * n * (4 + 3 * k) * d * d + 14 * c["batch"] * _pairs(c["seq"], c["window"]) * d
        return {"bytes": by, "flops": fl}
    if kind == "attn":
        b, s, h, hd = c["batch"], c["seq"], c["heads"], c["head_dim"]
        n, pairs = b * s * h, b * h * _pairs(s, c["window"])
        return {"bytes": n * hd * (4 * 2 + 3 * 2 + 4 * 4) + 2 * n * 2 * c["window"], "flops": 14 * pairs * hd}
    B, s = c["chains"], c["seq"]
    if kind == "hope":
        # per token 30 d^2 forward and 58 d^2 backward where the six memories share their factors inside a chunk
        return {"bytes": 4 * (4 * B * s * 64) + 2 * 4 * B * (-(-s // c["chunk"]) + 2) * 6 * 64 * 64,
                "flops": B * s * (30 + 58) * 64 * 64}
    d, mats = c.get("head_dim", 64), 2 if c["rule"] == "titans" else 1
    if kind == "exact":
        by, fl = _rule_work(B * s, d, mats, B * checkpoint_count(s, c["interval"]), 4, (39 if mats == 2 else 26) * d * d)
    else:
        by, fl = _rule_work(B * s, d, mats, B * (-(-s // c["chunk"]) + 1), 2 if kind == "chunk_bf16" else 4,
                            200704 if mats == 2 else 140000)
    return {"bytes": by, "flops": fl}


def tolerance(case):
    kind = case["kind"]
    if kind in ("decode", "prefill", "train", "chunk_bf16", "attn"):
        return {"rel": 1e-2}      # bf16 attention or bf16 tokens, fp32 accumulation
    if kind == "layer":
        return {"rel": 1.5e-2}    # projections, tokens and attention in bf16
    if kind == "hope":
        return {"rel": 1e-4}      # fp32, but the gates feed back into the recurrence
    return {"rel": 2e-5}          # fp32 sums over a chain
