"""The single-element gradients of a training step at the size the reference quotes its training rate for (d = 512, four levels,
512 tokens, vocabulary 32 000), against the same step in float64.  A gate bias's gradient is a sum over all tokens that cancels to
1e-2 of its terms and now and then to 1e-6, so that its relative error says nothing; its error over the sum of the terms'
magnitudes does.  The float64 step takes the attention's output as the device left it: bf16 roundings are not what is looked at."""
import math

import pytest
import torch
import torch.nn.functional as F

from nl_hecate_amd import cms_model as GM
from nl_hecate_amd.cms import ContextState, Pulse
from nl_hecate_amd.mag_layer import MemoryLevelParams
from nl_hecate_amd.memory_level import LevelConfig
from nl_hecate_amd.serving import GpuMAGParams
from tests.torch_mag_reference import titans

pytestmark = pytest.mark.gpu
HEADS, HD, LEVELS, SEQ, VOCAB, WINDOW = 8, 64, 4, 512, 32000, 512
GATES = ("alpha", "theta", "eta")


def random_model(seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    d = HEADS * HD
    normal = lambda *sh, std=1.0: torch.randn(*sh, generator=g, device="cuda") * std
    uniform = lambda lim, *sh: (torch.rand(*sh, generator=g, device="cuda") * 2 - 1) * lim
    w = lambda rows, cols: uniform(math.sqrt(6.0 / (rows + cols)), rows, cols)
    one = lambda x: torch.full((1,), x, device="cuda")
    levels = [MemoryLevelParams(w(d, d), w(d, d), w(d, d), uniform(0.05, 2 * d), one(-2.0), uniform(0.05, 2 * d), one(-3.0),
                                uniform(0.05, 2 * d), one(2.0)) for _ in range(LEVELS)]
    params = GpuMAGParams(normal(VOCAB, d), w(d, d), w(d, d), w(d, d), w(d, d), w(d, VOCAB), levels)
    memory = [normal(HEADS, HD * HD, std=0.05) for _ in range(LEVELS)]
    ids, targets = (torch.randint(0, VOCAB, (SEQ,), generator=g, device="cuda").tolist() for _ in range(2))
    return params, memory, ids, targets


def float64_terms(params, memory, ids, targets, attn_out):
    """What each token adds to the gradient of each level's gate biases: [levels][gate] -> [tokens]."""
    x = params.w_embed[torch.tensor(ids, device="cuda")].double()
    heads = lambda t: t.view(SEQ, HEADS, HD).transpose(0, 1)
    unit = lambda t: t / t.norm(dim=-1, keepdim=True).clamp_min(1e-8)
    chains, pre = [], []
    for lp in params.levels:
        k, v, q = unit(x @ lp.w_k.double().t()), x @ lp.w_v.double().t(), unit(x @ lp.w_q.double().t())
        kv = torch.cat([k, v], 1)
        a = [(kv @ getattr(lp, "w_" + n).double() + getattr(lp, "b_" + n).double()).requires_grad_() for n in GATES]
        pre.append(a)
        each = lambda t: t.expand(HEADS, SEQ)
        chains.append((heads(k), heads(v), heads(q), each(torch.sigmoid(a[0])), each(F.softplus(a[1])), each(torch.sigmoid(a[2]))))
    m0 = torch.cat(memory).double().view(-1, HD, HD)
    y, _, _ = titans(*(torch.cat(t) for t in zip(*chains)), m0, torch.zeros_like(m0))
    y = y.view(LEVELS, HEADS, SEQ, HD).sum(0).transpose(0, 1).reshape(SEQ, HEADS * HD) / math.sqrt(LEVELS)
    logits = (attn_out.double() * torch.sigmoid(y)) @ params.w_o.double().t() @ params.w_unembed.double()
    grads = torch.autograd.grad(F.cross_entropy(logits, torch.tensor(targets, device="cuda")), [t for a in pre for t in a])
    return [grads[3 * i:3 * i + 3] for i in range(LEVELS)]


def bias_errors(seed):
    """Each bias gradient's distance from float64 over the sum of its terms' magnitudes."""
    params, memory, ids, targets = random_model(seed)
    cfg = GM.ModelConfig(HEADS * HD, VOCAB, HEADS, HD, WINDOW, SEQ, [LevelConfig("titans", HEADS, HD) for _ in range(LEVELS)])
    _, cache = GM.gpu_cms_forward(params, cfg, ids, targets, Pulse(0, [True] * LEVELS), ContextState([m.clone() for m in memory]))
    grads = GM.gpu_cms_backward(params, cfg, cache)
    terms = float64_terms(params, memory, ids, targets, cache["attn_out"])
    return [(abs(getattr(lg, "d_b_" + n).double() - t.sum()) / t.abs().sum()).item()
            for lg, level in zip(grads.levels, terms) for n, t in zip(GATES, level)]


@pytest.mark.parametrize("seed", [1, 2])
def test_bias_gradients_against_the_sum_of_their_terms(seed):
    print(seed, flush=True)
    errors = bias_errors(seed)
    # a term comes out of some twenty fp32 products and sums in a row, each within 2^-23 of its own terms' magnitudes
    assert max(errors) <= 20 * 2 ** -23, errors
