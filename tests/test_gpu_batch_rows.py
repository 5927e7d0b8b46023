"""A row's bits do not depend on the batch around it: the BF16 experts, the FFN
block's shared MLP and Linear4Bit sum every output over the same ranges of K in
the same order, whether a call streams the weights (few rows) or runs the tiled
GEMM (many).  Rows of a large call are compared with the same rows in calls of
few rows, bit for bit.

The shapes: ranges of one 32-wide step (K <= 256), ranges that end inside a
64-wide stage, K ranges without a step (K / 32 not filling them), a last half
stage, and the Gemma widths; row counts around every tile height."""
import pytest
import torch

from hybridagent_amd import _lib, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    assert _lib.available(), "libw4a16moe.so must be built"
    return torch.device("cuda:0")


@pytest.mark.parametrize("H,I", [(160, 192), (288, 160), (544, 416), (2112, 352), (2816, 704)])
def test_bf16_experts_rows(dev, H, I):
    # one expert per token, segments of every tile height: 1 .. 300 rows
    rows = [1, 32, 33, 64, 65, 96, 97, 128, 129, 300]
    E = len(rows)
    g = torch.Generator(device=dev).manual_seed(41)
    gu = (torch.randn(E, 2 * I, H, generator=g, device=dev) / H ** 0.5).to(torch.bfloat16)
    dn = (torch.randn(E, H, I, generator=g, device=dev) / I ** 0.5).to(torch.bfloat16)
    idx = torch.repeat_interleave(torch.arange(E), torch.tensor(rows))
    idx = idx[torch.randperm(idx.numel(), generator=torch.Generator().manual_seed(42))][:, None].to(dev)
    M = idx.shape[0]
    x = synth.activations(M, H, seed=43, device=dev)
    w = torch.rand(M, 1, generator=g, device=dev) + 0.5
    whole = _lib.bf16_experts_forward(x, idx, w, gu, dn)
    for lo in range(0, M, 190):  # at most 192 routed rows stream the weights
        s = slice(lo, lo + 190)
        assert torch.equal(whole[s], _lib.bf16_experts_forward(x[s], idx[s], w[s], gu, dn)), f"rows from {lo}"


@pytest.mark.parametrize("H,Im,M", [(288, 2112, 1411), (2816, 1056, 300), (2816, 2112, 129), (2816, 2112, 481),
                                    (2816, 1120, 1025), (2816, 2112, 2048), (2816, 352, 2300),
                                    (2816, 352, 3000)])
def test_ffn_shared_mlp_rows(dev, H, Im, M):
    """The block with experts whose weights are all zero (q = 0): its output is norm3(norm1(mlp) + 0)."""
    I, E, G = 192, 4, 32
    g = torch.Generator(device=dev).manual_seed(51)
    lin = lambda o, i: (torch.randn(o, i, generator=g, device=dev) / i ** 0.5).to(torch.bfloat16)
    one = torch.ones(H, dtype=torch.bfloat16, device=dev)
    zero = lambda *s: torch.full(s, -2004318072, dtype=torch.int32, device=dev)  # 0x88888888: q = 0
    sc = lambda *s: torch.full(s, 0.01, dtype=torch.bfloat16, device=dev)
    rw = synth.router_weights(E, H, seed=52, device=dev)
    gate, up, down = lin(Im, H), lin(Im, H), lin(H, Im)
    gu, gus, dn, dns = zero(E, 2 * I, H // 8), sc(E, 2 * I, -(-H // G)), zero(E, H, I // 8), sc(E, H, -(-I // G))
    res, att = synth.activations(M, H, seed=53, device=dev), synth.activations(M, H, seed=54, device=dev)

    def block(s):
        return _lib.ffn_block(res[s], att[s], one, one, gate, up, down, one, rw.scale, rw.scalar_root, rw.proj,
                              rw.per_expert_scale, one, gu, gus, dn, dns, one, one, one[:1], 1e-6, 2, G)

    whole = block(slice(0, M))
    # 64 rows stream the weights on fragment-order rows, 16 on row-major ones
    for lo, n in [(0, 64), (M // 2, 64), (M - 64, 64), (M - 16, 16), (M - 1, 1)]:
        assert torch.equal(whole[lo:lo + n], block(slice(lo, lo + n))), f"rows from {lo}"


# K: one to four ranges of every length, a range without a tile (2112), tiles of 1 to 4 32-wide chunks last, ranges
# whose tiles lie apart (3200, 9216); M at N = 2816: every tile height, 1 .. 6 row blocks, whole and not
@pytest.mark.parametrize("K", [160, 256, 352, 512, 672, 704, 992, 1056, 2048, 2112, 2816, 3072, 3200, 9216])
@pytest.mark.parametrize("M,N,G", [(330, 2816, 32), (700, 2816, 128), (1201, 2816, 32), (1800, 2816, 64),
                                   (2300, 2816, 32), (4096, 2816, 128), (700, 1357, 32)])
def test_linear4bit_rows(dev, K, M, N, G):
    p = synth.packed_int4((N, K), 61, dev)
    s = synth.group_scales((N, K), G, 62, dev)
    x = synth.activations(M, K, 63, dev)
    whole = _lib.linear(x, p, s, None, G)
    for lo, n in [(0, 300), (M // 2, 17), (M - 300, 300), (M - 1, 1)]:  # at most 900e3 outputs stream the weights
        assert torch.equal(whole[lo:lo + n], _lib.linear(x[lo:lo + n], p, s, None, G)), f"rows from {lo}"
