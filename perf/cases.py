"""The calls whose speed this repository is about, with their inputs, the work they cannot do
without, and what another correct implementation may differ by.

Every case is one call of a public entry point:

* ``layer``      router + W4A16 experts (``_lib.moe_layer_forward``)
* ``latent``     the same with the residual add and the next layer's norm, one layer of the latent
                 loop (``_lib.moe_layer_forward_add_norm``)
* ``experts``    ``Gemma4TextExperts4Bit.forward`` on a routing the caller has
* ``ffn``        the post-attention FFN block of a decoder layer (``backends.ffn_moe_4bit_step``)
* ``bf16``       the unquantised experts (``backends.bf16_experts_fast_forward``)
* ``linear``     ``Linear4Bit.forward``
* ``hybridlink`` the latent map of the last hidden state (``_lib.hybridlink``)

at the Gemma-4-26B-A4B shape (hidden 2816, 128 experts, top-8, expert intermediate 704, shared MLP
2112) and, among the drawn cases, at a small one.  ``T`` is the number of tokens of the call:
1 is a chat's decode step, up to 64 a served batch, up to 256 a large batch or a short prompt,
beyond that a prompt's prefill.  Group size 32 is the released checkpoints', 128 the benchmark's.
"""
import math
from types import SimpleNamespace

import torch
import torch.nn.functional as F

from hybridagent_amd import _lib, backends, quantization

EPS = 1e-6
GEMMA = {"E": 128, "H": 2816, "I": 704, "k": 8}
SMALL = {"E": 32, "H": 2048, "I": 512, "k": 4}


def listed():
    return [
        # a chat's decode step through one MoE layer: launches and latency
        {"name": "layer_decode_1", "kind": "layer", "T": 1, "G": 128, "tiled": True, "skew": 0.0, **GEMMA},
        # a served batch's decode step on the released checkpoints' group size: streams nearly every expert
        {"name": "experts_decode_64", "kind": "experts", "T": 64, "G": 32, "tiled": True, "skew": 0.0, **GEMMA},
        # a large batch, or a short prompt, between the decode and prefill kernels; odd size
        {"name": "experts_batch_193", "kind": "experts", "T": 193, "G": 32, "tiled": True, "skew": 0.0, **GEMMA},
        # a prompt on a model loaded without the tiled copies, skewed routing, ragged size
        {"name": "experts_prompt_777", "kind": "experts", "T": 777, "G": 32, "tiled": False, "skew": 1.1, **GEMMA},
        # the benchmark's prefill: a long prompt, skewed routing, some experts without a row
        {"name": "layer_prefill_4096", "kind": "layer", "T": 4096, "G": 128, "tiled": True, "skew": 1.1, **GEMMA},
        # the FFN half of a decoder layer at a chat's decode step, as patch_ffn_4bit runs it
        {"name": "ffn_decode_1", "kind": "ffn", "T": 1, "G": 32, "tiled": True, "skew": 0.0, "Im": 2112, **GEMMA},
        # the same block at a prompt's prefill: here the shared bf16 MLP has work of its own
        {"name": "ffn_prefill_2048", "kind": "ffn", "T": 2048, "G": 32, "tiled": True, "skew": 1.1, "Im": 2112,
         **GEMMA},
        # the unquantised experts at a small served batch
        {"name": "bf16_decode_8", "kind": "bf16", "T": 8, "skew": 0.0, **GEMMA},
        # and at a prompt, skewed routing, ragged size
        {"name": "bf16_prompt_1031", "kind": "bf16", "T": 1031, "skew": 1.1, **GEMMA},
        # the dense 4-bit linear at decode sizes
        {"name": "linear_decode_4", "kind": "linear", "T": 4, "G": 128, "K": 2816, "N": 2816, "bias": False},
        # and at a prompt, with a bias
        {"name": "linear_prompt_2048", "kind": "linear", "T": 2048, "G": 32, "K": 2816, "N": 2816, "bias": True},
        # the latent loop's map at its batch of 32
        {"name": "hybridlink_32", "kind": "hybridlink", "T": 32, "H": 2816},
    ]


def _tokens(rng, most):
    """A token count spread over the logarithm of 1 .. most."""
    return min(most, max(1, int(round(math.exp(rng.uniform(0.0, math.log(most)))))))


def draw(rng):
    """One more case of these ranges, not one of the listed."""
    known = [{n: v for n, v in c.items() if n != "name"} for c in listed()]
    while True:
        case = _draw(rng)
        if case not in known:
            return case


def _draw(rng):
    kind = rng.choice(["layer", "latent", "experts", "experts", "ffn", "ffn", "bf16", "bf16", "linear", "linear",
                       "hybridlink"])
    if kind == "linear":
        # the benchmark's dense shapes, or any other between them
        K, N = rng.choice([(2816, 2816), (2816, 1408), (704, 2816),
                           (32 * rng.randint(22, 88), rng.randint(704, 2816))])
        return {"kind": kind, "T": _tokens(rng, 4096), "G": rng.choice([32, 128]), "K": K, "N": N,
                "bias": rng.random() < 0.3}
    if kind == "hybridlink":
        return {"kind": kind, "T": _tokens(rng, 256), "H": rng.choice([2816, 2816, 32 * rng.randint(64, 87)])}
    case = {"kind": kind, "skew": rng.choice([0.0, 1.1]), **(SMALL if rng.random() < 0.2 else GEMMA)}
    if kind == "bf16":
        case["T"] = _tokens(rng, 1031)
        return case
    case["T"] = _tokens(rng, {"layer": 4096, "latent": 64, "experts": 4096, "ffn": 2048}[kind])
    case["G"] = rng.choice([32, 32, 128])
    case["tiled"] = rng.random() < 0.7
    if kind == "ffn":
        case["Im"] = 32 * rng.randint(33, 66)
    return case


# ---------------------------------------------------------------------------- inputs


class _Gen:
    """Seeded values on the GPU."""

    def __init__(self, seed, device="cuda"):
        self.g = torch.Generator(device=device).manual_seed(seed)
        self.dev = device

    def normal(self, *shape, std=1.0, mean=0.0):
        t = torch.randn(*shape, generator=self.g, device=self.dev, dtype=torch.float32)
        return t.mul_(std).add_(mean).to(torch.bfloat16)

    def words(self, *shape):
        """Packed int4 weights: uniform nibbles, so uniform 32-bit words."""
        return torch.randint(-(2 ** 31), 2 ** 31, shape, generator=self.g, device=self.dev,
                             dtype=torch.int64).to(torch.int32)

    def scales(self, *shape):
        t = torch.rand(*shape, generator=self.g, device=self.dev, dtype=torch.float32)
        return t.mul_(0.015).add_(0.005).to(torch.bfloat16)

    def gumbel(self, *shape):
        u = torch.rand(*shape, generator=self.g, device=self.dev, dtype=torch.float32).clamp_(1e-7, 1 - 1e-7)
        return -torch.log(-torch.log(u))


def _expert_bias(g, E, skew):
    """log-probabilities of the experts: flat, or Zipf(skew) over a random order."""
    rank = torch.randperm(E, generator=g.g, device=g.dev).float() + 1.0
    return -skew * torch.log(rank)


def _inputs(case, seed):
    """Everything the call and its weights are made of, from the seed alone."""
    g = _Gen(seed)
    c = SimpleNamespace(**case)
    s = SimpleNamespace(case=case)
    if c.kind == "linear":
        s.x = g.normal(c.T, c.K)
        s.packed, s.scale = g.words(c.N, c.K // 8), g.scales(c.N, -(-c.K // c.G))
        s.bias = g.normal(c.N, std=0.1) if c.bias else None
        return s
    if c.kind == "hybridlink":
        std = c.H ** -0.5
        s.x = g.normal(c.T, c.H)
        s.ln1w, s.ln1b = g.normal(c.H, std=0.05, mean=1.0), g.normal(c.H, std=0.02)
        s.p1w, s.p1b = g.normal(c.H, c.H, std=std), g.normal(c.H, std=0.02)
        s.p2w, s.p2b = g.normal(c.H, c.H, std=std), g.normal(c.H, std=0.02)
        s.ln2w, s.ln2b = g.normal(c.H, std=0.05, mean=1.0), g.normal(c.H, std=0.02)
        return s
    E, H, I, k, T = c.E, c.H, c.I, c.k, c.T
    # the experts' input is a normalised row, the router's a residual row
    s.x = g.normal(T, H)
    if c.kind in ("experts", "bf16"):
        # a routing the caller has: top-k of noisy expert log-probabilities
        noisy = _expert_bias(g, E, c.skew)[None, :] + g.gumbel(T, E)
        val, s.idx = torch.topk(noisy, k, dim=-1)
        s.w = torch.softmax(val, dim=-1)
    else:
        s.residual = g.normal(T, H)
        # logits ~ N(bias, 1): the router's normalised input has unit norm, its coordinate 0 carries the bias
        proj = torch.randn(E, H, generator=g.g, device=g.dev)
        if c.skew:
            s.residual[:, 0] = 8.0
            proj[:, 0] = _expert_bias(g, E, c.skew) / (8.0 * H ** -0.5)
        s.proj = proj.to(torch.bfloat16)
        s.router_scale = g.normal(H, std=0.02, mean=1.0)
        s.pes = g.normal(E, std=0.02, mean=1.0)
        s.root = H ** -0.5
    if c.kind == "bf16":
        s.gu = torch.stack([g.normal(2 * I, H, std=0.02) for _ in range(E)])
        s.dn = torch.stack([g.normal(H, I, std=0.02) for _ in range(E)])
        return s
    s.gu_p = torch.stack([g.words(2 * I, H // 8) for _ in range(E)])
    s.dn_p = torch.stack([g.words(H, I // 8) for _ in range(E)])
    s.gu_s, s.dn_s = g.scales(E, 2 * I, -(-H // c.G)), g.scales(E, H, -(-I // c.G))
    if c.kind == "latent":
        s.norm = g.normal(H, std=0.05, mean=1.0)
    if c.kind == "ffn":
        s.attn = g.normal(T, H)
        s.lnw = [g.normal(H, std=0.05, mean=1.0) for _ in range(6)]
        s.gate, s.up = g.normal(c.Im, H, std=0.02), g.normal(c.Im, H, std=0.02)
        s.down = g.normal(H, c.Im, std=0.02)
        s.layer_scalar = torch.full((1,), 0.75, dtype=torch.bfloat16, device=g.dev)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "linear":
        s.mod = quantization.Linear4Bit(case["K"], case["N"], bias=case["bias"], group_size=case["G"]).to("cuda")
        s.mod.weight_packed.copy_(s.packed)
        s.mod.weight_scale.copy_(s.scale)
        if s.bias is not None:
            s.mod.bias.data.copy_(s.bias)
    elif kind == "bf16":
        s.mod = SimpleNamespace(gate_up_proj=s.gu, down_proj=s.dn)
    elif kind != "hybridlink":
        # the experts module of a loaded checkpoint, with or without its tiled copies
        cfg = SimpleNamespace(num_experts=case["E"], hidden_size=case["H"], moe_intermediate_size=case["I"])
        with torch.device("cuda"):
            s.mod = quantization.Gemma4TextExperts4Bit(cfg, group_size=case["G"])
        for name, t in (("gate_up_packed", s.gu_p), ("gate_up_scale", s.gu_s), ("down_packed", s.dn_p),
                        ("down_scale", s.dn_s)):
            getattr(s.mod, name).copy_(t)
        del s.gu_p, s.gu_s, s.dn_p, s.dn_s
        if case["tiled"]:
            s.mod.tile_weights()
    return s


def run(s):
    case = s.case
    kind = case["kind"]
    m = getattr(s, "mod", None)
    if kind == "linear":
        return m(s.x)
    if kind == "hybridlink":
        return _lib.hybridlink(s.x, s.ln1w, s.ln1b, s.p1w, s.p1b, s.p2w, s.p2b, s.ln2w, s.ln2b)
    if kind == "bf16":
        return backends.bf16_experts_fast_forward(m, s.x, s.idx, s.w)
    if kind == "experts":
        return m(s.x, s.idx, s.w)
    ew = (m.gate_up_packed, m.gate_up_scale, m.down_packed, m.down_scale)
    if kind == "layer":
        out, w, idx = _lib.moe_layer_forward(s.residual, s.router_scale, s.root, s.proj, s.pes, EPS, case["k"], s.x,
                                             *ew)
        return {"out": out, "w": w, "idx": idx}
    if kind == "latent":
        h, y, out, w, idx = _lib.moe_layer_forward_add_norm(s.residual, s.router_scale, s.root, s.proj, s.pes, EPS,
                                                            case["k"], s.x, *ew, s.norm, EPS)
        return {"h": h, "y": y, "out": out, "w": w, "idx": idx}
    ln = s.lnw
    return backends.ffn_moe_4bit_step(s.residual, s.attn, ln[0], ln[1], s.gate, s.up, s.down, ln[2], s.router_scale,
                                      s.root, s.proj, s.pes, ln[3], *ew, ln[4], ln[5], s.layer_scalar, EPS,
                                      case["k"])


# ---------------------------------------------------------------------------- work


def _experts_hit(E, k, T):
    """Distinct experts that T tokens of top-k routing hit, for a flat routing."""
    return E * (1.0 - (1.0 - k / E) ** T)


def work(case):
    T, kind = case["T"], case["kind"]
    if kind == "linear":
        K, N = case["K"], case["N"]
        return {"bytes": N * K // 2 + N * -(-K // case["G"]) * 2 + 2 * T * (K + N) + (2 * N if case["bias"] else 0),
                "flops": 2 * T * K * N}
    H = case["H"]
    if kind == "hybridlink":
        return {"bytes": 4 * H * H + 12 * H + 4 * T * H, "flops": 4 * T * H * H}
    E, I, k = case["E"], case["I"], case["k"]
    U = _experts_hit(E, k, T)
    flops = 2 * T * k * 3 * H * I
    if kind == "bf16":
        return {"bytes": int(U * 6 * H * I) + 4 * T * H + 12 * T * k, "flops": flops}
    G = case["G"]
    per_expert = 3 * H * I // 2 + 2 * (2 * I * -(-H // G) + H * -(-I // G))
    nbytes = int(U * per_expert) + 4 * T * H
    if kind == "experts":
        return {"bytes": nbytes + 12 * T * k, "flops": flops}
    nbytes += 2 * E * H + 2 * H + 2 * E
    flops += 2 * T * E * H
    if kind == "ffn":
        Im = case["Im"]
        return {"bytes": nbytes + 6 * Im * H + 14 * H + 2 * T * H, "flops": flops + 6 * T * H * Im}
    nbytes += 2 * T * H + 12 * T * k
    return {"bytes": nbytes + (4 * T * H if kind == "latent" else 0), "flops": flops}


def tolerance(case):
    # bf16 results of bf16 products summed in 32 bits: the sums' order moves single results by one rounding of
    # bf16.  The gated product, the combine and the norms hold several such roundings in a row.
    kind = case["kind"]
    if kind == "linear":
        return {"rel": 4e-3, "max": 0.05}
    if kind == "hybridlink":
        return {"rel": 6e-3, "max": 0.05}
    if kind == "ffn":
        return {"rel": 6e-3, "max": 0.1}
    if kind in ("layer", "latent"):
        return {"rel": 1e-2, "max": 0.15, "differ": 2e-3}
    return {"rel": 1e-2, "max": 0.15}


# ---------------------------------------------------------------------------- 64-bit results


def _dequant64(packed, scale, G):
    """The weights a packed matrix stands for: bf16(q * s), as the format defines them."""
    K = packed.shape[-1] * 8
    sh = torch.arange(0, 32, 4, dtype=torch.int32, device=packed.device)
    q = (((packed.unsqueeze(-1) >> sh) & 15) - 8).reshape(*packed.shape[:-1], K)
    s = scale.repeat_interleave(G, dim=-1)[..., :K]
    return (q.float() * s.float()).to(torch.bfloat16).double()


def _gelu_tanh(x):
    return F.gelu(x, approximate="tanh")


def _rms(x, w=None):
    x = x.double()
    y = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS)
    return y if w is None else y * w.double()


def _bf(x):
    return x.to(torch.bfloat16).double()


def _route(s, rows, k):
    """(weights, indices): the router picks by bf16 logits of bf16 inputs, lower index first among equals."""
    r = _bf(_bf(_bf(_rms(rows)) * s.router_scale.double()) * s.root)
    lg = _bf(r @ s.proj.double().t())
    E = lg.shape[-1]
    # equal logits: distinct keys one part in 2^40 apart, below any gap between two bf16 values
    idx = torch.topk(lg - torch.arange(E, device=lg.device) * 2.0 ** -40, k, dim=-1).indices
    p = torch.gather(torch.softmax(lg, -1), -1, idx)
    return p / p.sum(-1, keepdim=True) * s.pes.double()[idx], idx


def _experts64(x, idx, w, weights_of, I):
    """sum_j w[t, j] * down(gelu(gate) * up) over the experts hit, all in 64 bits."""
    out = torch.zeros(x.shape, dtype=torch.float64, device=x.device)
    xd = x.double()
    for e in torch.unique(idx).tolist():
        t, j = torch.where(idx == e)
        gu, dn = weights_of(e)
        h = xd[t] @ gu.t()
        y = (_gelu_tanh(h[:, :I]) * h[:, I:]) @ dn.t()
        out.index_add_(0, t, y * w[t, j].double()[:, None])
    return out


def exact(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "linear":
        y = s.x.double() @ _dequant64(s.packed, s.scale, case["G"]).t()
        return y if s.bias is None else y + s.bias.double()
    if kind == "hybridlink":
        d = lambda n: getattr(s, n).double()
        H = case["H"]
        a = F.layer_norm(s.x.double(), (H,), d("ln1w"), d("ln1b"), 1e-5)
        a = F.gelu(a @ d("p1w").t() + d("p1b")) @ d("p2w").t() + d("p2b")
        return F.layer_norm(s.x.double() + a, (H,), d("ln2w"), d("ln2b"), 1e-5)
    I, k = case["I"], case["k"]
    if kind == "bf16":
        return _experts64(s.x, s.idx, s.w, lambda e: (s.gu[e].double(), s.dn[e].double()), I)
    weights_of = lambda e: (_dequant64(s.gu_p[e], s.gu_s[e], case["G"]), _dequant64(s.dn_p[e], s.dn_s[e], case["G"]))
    if kind == "experts":
        return _experts64(s.x, s.idx, s.w, weights_of, I)
    if kind in ("layer", "latent"):
        w, idx = _route(s, s.residual, k)
        out = _experts64(s.x, idx, w, weights_of, I)
        if kind == "layer":
            return {"out": out, "w": w, "idx": None}
        h = s.residual.double() + out
        return {"h": h, "y": _rms(h, s.norm), "out": out, "w": w, "idx": None}
    ln = s.lnw
    res = s.residual.double() + _rms(s.attn, ln[0])
    hff = _rms(res, ln[1])
    mlp = (_gelu_tanh(hff @ s.gate.double().t()) * (hff @ s.up.double().t())) @ s.down.double().t()
    # the router reads the bf16 residual row, as the block's other rounding points leave it
    w, idx = _route(s, _bf(s.residual.double() + _bf(_rms(s.attn, ln[0]))), k)
    moe = _experts64(_rms(res, ln[3]), idx, w, weights_of, I)
    comb = _rms(_rms(mlp, ln[2]) + _rms(moe, ln[4]), ln[5])
    return (res + comb) * s.layer_scalar.double()
