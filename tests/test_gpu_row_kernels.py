"""The row kernels built per 16-byte chunks of a thread (H <= 2048, 4096, 6144, 8192)
and the FFN block's last launch with the combine inside: a token's row equals,
bit for bit, the same token's in calls of four (32 routed rows: the fused down +
combine, then the block's last launch on its output), at each chunk count, and
at top_k = 9, which combines in a launch of its own.  The norms against torch."""
import math

import pytest
import torch
import torch.nn.functional as F

from hybridagent_amd import _lib, synth

pytestmark = pytest.mark.gpu

# rows of one chunk and less, edges of one, two, three and four chunks per thread
WIDTHS = [256, 2048, 2080, 2816, 4096, 4128, 6144, 8192]


@pytest.mark.parametrize("H", WIDTHS)
@pytest.mark.parametrize("k", [8, 9])
def test_ffn_post_combines_bit_identical(H, k):
    dev = torch.device("cuda:0")
    E, I, Im, G, M = 16, 64, 96, 32, 12
    g = torch.Generator().manual_seed(H + k)
    nrm = lambda: (1 + 0.1 * torch.randn(H, generator=g)).to(torch.bfloat16).to(dev)
    lin = lambda o, i: (torch.randn(o, i, generator=g) / math.sqrt(i)).to(torch.bfloat16).to(dev)
    w = synth.moe_weights(E, H, I, G, seed=3, device=dev)
    rw = synth.router_weights(E, H, seed=4, device=dev)
    res, att = synth.activations(M, H, 5, dev), synth.activations(M, H, 6, dev)
    tail = (nrm(), nrm(), lin(Im, H), lin(Im, H), lin(H, Im), nrm(), nrm(), H ** -0.5, rw.proj, rw.per_expert_scale,
            nrm(), w.gate_up_packed, w.gate_up_scale, w.down_packed, w.down_scale, nrm(), nrm(),
            torch.full((1,), 0.5, dtype=torch.bfloat16, device=dev), 1e-6, k, G)
    y = _lib.ffn_block(res, att, *tail)
    step = 4 if k == 8 else 3
    for m in range(0, M, step):
        assert torch.equal(_lib.ffn_block(res[m:m + step], att[m:m + step], *tail), y[m:m + step]), f"rows {m}.."


# The shared MLP's rows in fragment order from 17 rows on (row tiles of 2 and 4,
# partial last tiles), and row-major where they don't fit (top_k 1;
# 2 at the wide Im): every row as in calls of 16 rows, which never use that order.
@pytest.mark.parametrize("M", [17, 31, 32, 33, 48, 63, 64])
@pytest.mark.parametrize("H,Im", [(256, 96), (2816, 2112), (512, 1056), (4128, 96), (8192, 96)])
@pytest.mark.parametrize("k", [1, 2, 8])
def test_ffn_fragment_rows_bit_identical(M, H, Im, k):
    dev = torch.device("cuda:0")
    E, I, G = 16, 64, 32
    g = torch.Generator().manual_seed(M + H + k)
    nrm = lambda: (1 + 0.1 * torch.randn(H, generator=g)).to(torch.bfloat16).to(dev)
    lin = lambda o, i: (torch.randn(o, i, generator=g) / math.sqrt(i)).to(torch.bfloat16).to(dev)
    w = synth.moe_weights(E, H, I, G, seed=3, device=dev)
    rw = synth.router_weights(E, H, seed=4, device=dev)
    res, att = synth.activations(M, H, 5, dev), synth.activations(M, H, 6, dev)
    tail = (nrm(), nrm(), lin(Im, H), lin(Im, H), lin(H, Im), nrm(), nrm(), H ** -0.5, rw.proj, rw.per_expert_scale,
            nrm(), w.gate_up_packed, w.gate_up_scale, w.down_packed, w.down_scale, nrm(), nrm(),
            torch.full((1,), 0.5, dtype=torch.bfloat16, device=dev), 1e-6, k, G)
    y = _lib.ffn_block(res, att, *tail)
    for m in range(0, M, 16):
        assert torch.equal(_lib.ffn_block(res[m:m + 16], att[m:m + 16], *tail), y[m:m + 16]), f"rows {m}.."


@pytest.mark.parametrize("H", WIDTHS)
def test_norms(H):
    dev = torch.device("cuda:0")
    x, d = synth.activations(5, H, 7, dev), synth.activations(5, H, 8, dev)
    w = (1 + 0.1 * torch.randn(H, generator=torch.Generator().manual_seed(9))).to(torch.bfloat16).to(dev)
    h, y = _lib.add_rms_norm(x, w, 1e-6, d)
    assert torch.equal(h, x + d)
    ref = F.rms_norm(h.double(), (H,), w.double(), 1e-6)
    # one rounding to bf16 (half a unit: 2^-8), and fp32 sums of H squares
    assert ((y.double() - ref).abs() <= 2.0 ** -8 * ref.abs() * (1 + 2.0 ** -7)).all()


def _unit(g, *shape):
    return (1 + 0.1 * torch.randn(*shape, generator=g, device=g.device)).to(torch.bfloat16)


@pytest.mark.parametrize("H", WIDTHS)
def test_hybridlink_rows(H):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(H)
    x = synth.activations(5, H, 10, dev)
    lin = lambda: (torch.randn(H, H, generator=g, device=dev) / math.sqrt(H)).to(torch.bfloat16)
    bias = lambda: (0.1 * torch.randn(H, generator=g, device=dev)).to(torch.bfloat16)
    l1w, l1b, p1, b1, p2, b2, l2w, l2b = _unit(g, H), bias(), lin(), bias(), lin(), bias(), _unit(g, H), bias()
    got = _lib.hybridlink(x, l1w, l1b, p1, b1, p2, b2, l2w, l2b).double()
    rb = lambda t: t.to(torch.bfloat16).double()
    a = rb(F.layer_norm(x.double(), (H,), l1w.double(), l1b.double()))
    a = rb(F.gelu(rb(a @ p1.double().t() + b1.double())))
    r = rb(x.double() + rb(a @ p2.double().t() + b2.double()))
    ref = F.layer_norm(r, (H,), l2w.double(), l2b.double())
    # an input of the last norm may have rounded the other way: four bf16 units (2^-8 of it, or of the projection
    # before it) through it, and the output's own rounding
    rstd = 1 / torch.sqrt(r.var(-1, unbiased=False, keepdim=True) + 1e-5)
    big = torch.maximum(torch.maximum(x.double().abs(), (r - x.double()).abs()), r.abs())
    assert ((got - ref).abs() <= 4 * 2.0 ** -7 * big * rstd * l2w.double().abs() + 2.0 ** -7 * ref.abs()).all()


@pytest.mark.parametrize("H", WIDTHS)
def test_layer_add_norm_rows(H):
    # 96 routed rows: the combine, the add and the norm in one launch, against the separate calls
    dev = torch.device("cuda:0")
    E, I, G, M, k = 16, 64, 32, 12, 8
    rw = synth.router_weights(E, H, seed=4, device=dev)
    w = synth.moe_weights(E, H, I, G, seed=3, device=dev)
    norm_w = _unit(torch.Generator(device=dev).manual_seed(H), H)
    h = synth.activations(M, H, 5, dev)
    xin = _lib.add_rms_norm(h, norm_w, 1e-6)[1]
    args = (h, rw.scale, rw.scalar_root, rw.proj, rw.per_expert_scale, rw.eps, k, xin, w.gate_up_packed,
            w.gate_up_scale, w.down_packed, w.down_scale)
    out, tw, idx = _lib.moe_layer_forward(*args, group_size=G)
    h_ref, y_ref = _lib.add_rms_norm(h, norm_w, 1e-6, delta=out)
    h2, y2, out2, tw2, idx2 = _lib.moe_layer_forward_add_norm(*args, norm_w, 1e-6, group_size=G)
    assert torch.equal(idx2, idx) and torch.equal(tw2, tw)
    assert torch.equal(out2, out) and torch.equal(h2, h_ref) and torch.equal(y2, y_ref)
