"""The prefill-size bf16 GEMMs (kernels_gemm_bf16.hip) through the entry points
that reach them: the BF16 experts on segments around every tile height, and
the FFN block's shared MLP at row counts around the dense tiles' edges, both at
widths whose last k stage is whole (K % 64 == 0) and half (K % 64 == 32) and
whose last column tile is partial.

Reference: float64 products of the bf16 operands, rounded to bf16 where the
kernels round.  A sum of K products in fp32 is off by at most K 2^-24 of the
sum of their magnitudes (every order); the bounds below add that to one
rounding of the output, and double it for what a flipped intermediate rounding
(one bf16 ulp of one of I inputs of the second product) moves."""
import math

import pytest
import torch
import torch.nn.functional as F

from hybridagent_amd import _lib, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    assert _lib.available(), "libw4a16moe.so must be built"
    return torch.device("cuda:0")


def _bf(x):
    return x.to(torch.bfloat16).double()


def _mlp64(x, gate, up, down):
    """(down(bf16(bf16(gelu(gate)) * up)), row-wise bound) in float64 on bf16 operands."""
    g, u = _bf(x @ gate.t()), _bf(x @ up.t())
    inter = _bf(_bf(F.gelu(g, approximate="tanh")) * u)
    y = inter @ down.t()
    # every input of the second product may have rounded the other way: one bf16 ulp (2^-8 of it) each, at most
    # their root sum of squares times 4, and the output's own rounding
    slack = 4 * 2.0 ** -8 * torch.sqrt(inter.pow(2) @ down.pow(2).t()) + 2.0 ** -8 * y.abs()
    return y, slack


# rows of the experts' segments: every tile height's edges, an empty expert, more than one 128-row tile
ROWS = [1, 31, 32, 33, 64, 65, 0, 95, 96, 97, 127, 128, 129, 160, 257, 2]


@pytest.mark.parametrize("H,I", [(256, 192), (160, 160), (288, 416), (2816, 704)])
def test_bf16_experts_segments(dev, H, I):
    E = len(ROWS)
    g = torch.Generator(device=dev).manual_seed(11)
    gu = (torch.randn(E, 2 * I, H, generator=g, device=dev) / math.sqrt(H)).to(torch.bfloat16)
    dn = (torch.randn(E, H, I, generator=g, device=dev) / math.sqrt(I)).to(torch.bfloat16)
    # one expert per token, in a random order
    idx = torch.repeat_interleave(torch.arange(E), torch.tensor(ROWS))
    idx = idx[torch.randperm(idx.numel(), generator=torch.Generator().manual_seed(12))]
    M = idx.numel()
    x = synth.activations(M, H, seed=13, device=dev)
    # a second slot without an expert, so that the routed rows pass the streaming kernel's range
    idx2 = torch.stack([idx, torch.full_like(idx, E)], 1).to(dev)
    w = torch.ones(M, 2, device=dev)
    got = _lib.bf16_experts_forward(x, idx2, w, gu, dn).double()
    for e in range(E):
        t = (idx == e).nonzero()[:, 0].to(dev)
        if t.numel() == 0:
            continue
        ref, slack = _mlp64(x[t].double(), gu[e, :I].double(), gu[e, I:].double(), dn[e].double())
        assert ((got[t] - ref).abs() <= slack).all(), f"expert {e} of {ROWS[e]} rows"


# at most 192 routed rows: the streaming kernel's chunks of 16, 32 and 64 rows
@pytest.mark.parametrize("rows", [[3, 15, 16, 17, 0, 2, 33, 40], [1, 31, 32, 33, 40, 0], [63, 64, 65]])
def test_bf16_experts_streamed_segments(dev, rows):
    E, H, I = len(rows), 256, 160
    g = torch.Generator(device=dev).manual_seed(31)
    gu = (torch.randn(E, 2 * I, H, generator=g, device=dev) / math.sqrt(H)).to(torch.bfloat16)
    dn = (torch.randn(E, H, I, generator=g, device=dev) / math.sqrt(I)).to(torch.bfloat16)
    idx = torch.repeat_interleave(torch.arange(E), torch.tensor(rows))
    idx = idx[torch.randperm(idx.numel(), generator=torch.Generator().manual_seed(32))]
    M = idx.numel()
    x = synth.activations(M, H, seed=33, device=dev)
    got = _lib.bf16_experts_forward(x, idx[:, None].to(dev), torch.ones(M, 1, device=dev), gu, dn).double()
    for e in range(E):
        t = (idx == e).nonzero()[:, 0].to(dev)
        if t.numel() > 0:
            ref, slack = _mlp64(x[t].double(), gu[e, :I].double(), gu[e, I:].double(), dn[e].double())
            assert ((got[t] - ref).abs() <= slack).all(), f"expert {e} of {rows[e]} rows"


# routed rows that are no multiple of four, all of them valid: the last row indices come in a 16-byte load that is
# partly past the plan's
@pytest.mark.parametrize("M,k", [(193, 1), (194, 1), (195, 1), (65, 3), (66, 3), (67, 3)])
def test_bf16_experts_last_rows(dev, M, k):
    E, H, I = 4, 256, 192
    g = torch.Generator(device=dev).manual_seed(61)
    gu = (torch.randn(E, 2 * I, H, generator=g, device=dev) / math.sqrt(H)).to(torch.bfloat16)
    dn = (torch.randn(E, H, I, generator=g, device=dev) / math.sqrt(I)).to(torch.bfloat16)
    gc = torch.Generator().manual_seed(62)
    idx = torch.stack([torch.randperm(E, generator=gc)[:k] for _ in range(M)])
    x = synth.activations(M, H, seed=63, device=dev)
    # one slot's weight at a time, so that every routed row of the last expert's segment shows
    for j in range(k):
        w = torch.zeros(M, k, device=dev)
        w[:, j] = 1.0
        got = _lib.bf16_experts_forward(x, idx.to(dev), w, gu, dn).double()
        for e in range(E):
            t = (idx[:, j] == e).nonzero()[:, 0].to(dev)
            ref, slack = _mlp64(x[t].double(), gu[e, :I].double(), gu[e, I:].double(), dn[e].double())
            assert ((got[t] - ref).abs() <= slack).all(), f"expert {e}, slot {j}"


@pytest.mark.parametrize("H,I", [(256, 192), (160, 160)])
def test_bf16_experts_two_slots_and_invalid(dev, H, I):
    # token-slot gathers (row / top_k) and slots without an expert, against the same routing on fp64
    E, M, k = 8, 700, 3
    g = torch.Generator(device=dev).manual_seed(21)
    gu = (torch.randn(E, 2 * I, H, generator=g, device=dev) / math.sqrt(H)).to(torch.bfloat16)
    dn = (torch.randn(E, H, I, generator=g, device=dev) / math.sqrt(I)).to(torch.bfloat16)
    gc = torch.Generator().manual_seed(22)
    idx = torch.stack([torch.randperm(E, generator=gc)[:k] for _ in range(M)])
    idx[::5, 1] = E
    idx[::7, 2] = -1
    x = synth.activations(M, H, seed=23, device=dev)
    w = (torch.rand(M, k, generator=gc) + 0.1).to(dev)
    got = _lib.bf16_experts_forward(x, idx.to(dev), w, gu, dn).double()
    ref, slack = torch.zeros(M, H, dtype=torch.float64, device=dev), torch.zeros(M, H, dtype=torch.float64, device=dev)
    for e in range(E):
        t, j = torch.where(idx == e)
        t, j = t.to(dev), j.to(dev)
        y, s = _mlp64(x[t].double(), gu[e, :I].double(), gu[e, I:].double(), dn[e].double())
        wj = _bf(w[t, j])[:, None]
        # dn, its weighted product and the sum round once each
        ref.index_add_(0, t, y * wj)
        slack.index_add_(0, t, (s + 3 * 2.0 ** -8 * y.abs()) * wj)
    assert ((got - ref).abs() <= slack + 2.0 ** -8 * ref.abs()).all()


# at H = 2816 the streams run up to 128 rows and, at Im = 1120 and 800, at 129 and 193; the others run tiles: their
# edges, half k stages (Im % 64 == 32) and rows enough for every tile height of the dense launch
@pytest.mark.parametrize("M,Im", [(65, 160), (81, 1056), (129, 1120), (193, 800), (257, 608), (300, 1056), (481, 2112),
                                  (700, 2112), (1025, 2112), (1700, 2112), (2047, 2112)])
def test_ffn_shared_mlp_rows(dev, M, Im):
    """The block with one expert whose weights are all zero (q = 0): its output is
    norm3(norm1(mlp) + 0), the shared MLP alone."""
    H, I, E, G = 2816, 192, 4, 32
    g = torch.Generator(device=dev).manual_seed(31)
    lin = lambda o, i: (torch.randn(o, i, generator=g, device=dev) / math.sqrt(i)).to(torch.bfloat16)
    one = torch.ones(H, dtype=torch.bfloat16, device=dev)
    zero = lambda *s: torch.full(s, -2004318072, dtype=torch.int32, device=dev)  # 0x88888888: q = 0
    sc = lambda *s: torch.full(s, 0.01, dtype=torch.bfloat16, device=dev)
    rw = synth.router_weights(E, H, seed=32, device=dev)
    gate, up, down = lin(Im, H), lin(Im, H), lin(H, Im)
    res, att = synth.activations(M, H, seed=33, device=dev), synth.activations(M, H, seed=34, device=dev)
    out = _lib.ffn_block(res, att, one, one, gate, up, down, one, rw.scale, rw.scalar_root, rw.proj,
                         rw.per_expert_scale, one, zero(E, 2 * I, H // 8), sc(E, 2 * I, -(-H // G)),
                         zero(E, H, I // 8), sc(E, H, -(-I // G)), one, one, one[:1], 1e-6, 2, G).double()
    rms = lambda t: t * torch.rsqrt(t.pow(2).mean(-1, keepdim=True) + 1e-6)
    r = _bf(res.double() + _bf(rms(att.double())))
    y, slack = _mlp64(_bf(rms(r)), gate.double(), up.double(), down.double())
    scale = torch.rsqrt(y.pow(2).mean(-1, keepdim=True) + 1e-6)
    ref = r + rms(_bf(rms(_bf(y))))
    # the MLP's slack through its norm (a factor of scale, and as much again from the row's mean square), the two
    # norms' roundings, the last sum's
    bound = 2 * slack * scale + 3 * 2.0 ** -8 * (y * scale).abs() + 2.0 ** -8 * ref.abs() + 2.0 ** -8
    bad = (out - ref).abs() > bound
    assert not bad.any(), f"{int(bad.sum())} of {bad.numel()} elements, worst {float(((out - ref).abs() / bound).max()):.2f} x the bound"
