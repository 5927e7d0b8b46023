"""The decode gate_up streamer's two-round form (more 16-row slots than half of the
chip's workgroups, at most two thirds): a token's row equals, bit for bit, the
same token's in calls of 32 tokens, which run one round -- on a plan the sort
wrote (moe_forward) and on the launch's own (moe_layer_forward at M * top_k
<= 1024), packed and tiled, either side of the slot range, whose slot count the
routing is made to hit on both."""
import pytest
import torch

from hybridagent_amd import _lib, synth

pytestmark = pytest.mark.gpu

E, H, I, K = 128, 2816, 256, 8


def _routing(M, n_full, seed):
    """[M, K] distinct experts per token with experts 0 .. n_full - 1 on 17 tokens or more each (two slots)."""
    g = torch.Generator().manual_seed(seed)
    want = torch.zeros(E, dtype=torch.long)
    want[:n_full] = 17
    left = M * K - int(want.sum())
    rest = E - n_full
    want[n_full:] = left // rest
    want[n_full:n_full + left % rest] += 1
    assert want[n_full:].max() <= 16 or n_full == 0, "the other experts keep one slot"
    # deal the experts' rows over the tokens in turn: distinct experts per token as long as no expert has M rows
    rows = torch.repeat_interleave(torch.arange(E), want)
    idx = rows.reshape(K, M).t().contiguous()
    assert all(len(set(r.tolist())) == K for r in idx)
    return idx[torch.randperm(M, generator=g)], int(((want + 15) // 16).sum())


@pytest.mark.parametrize("tiled", [False, True])
@pytest.mark.parametrize("G", [32, 128])
@pytest.mark.parametrize("M,n_full,slots", [(96, 0, 128), (120, 1, 129), (150, 20, 148), (180, 42, 170),
                                            (180, 43, 171), (200, 60, 188)])
def test_two_rounds_bit_identical(M, n_full, slots, G, tiled):
    dev = torch.device("cuda:0")
    w = synth.moe_weights(E, H, I, G, seed=81, device=dev)
    ew = (w.gate_up_packed, w.gate_up_scale, w.down_packed, w.down_scale)
    tiles = _lib.tile_experts(*ew, G) if tiled else None
    idx, n = _routing(M, n_full, 82)
    assert n == slots
    idx = idx.to(dev)
    wt = torch.rand(M, K, generator=torch.Generator().manual_seed(83)).to(dev)
    x = synth.activations(M, H, seed=84, device=dev)
    print(f"two rounds M={M} slots={slots} G={G} tiled={tiled}", flush=True)
    y = _lib.moe_forward(x, idx, wt, *ew, G, tiles=tiles)
    for m in range(0, M, 32):
        s = slice(m, m + 32)
        assert torch.equal(_lib.moe_forward(x[s], idx[s], wt[s], *ew, G, tiles=tiles), y[s]), f"rows {m}.."


# the two-round kernels of the other shapes: two and four k tiles per wavefront, the long-K loop (packed weights only)
@pytest.mark.parametrize("H,G,tiled", [(1024, 128, False), (1024, 32, False), (1024, 128, True), (1024, 32, True),
                                       (2048, 128, False), (2048, 32, False), (2048, 128, True), (2048, 32, True),
                                       (4096, 128, False)])
def test_two_rounds_other_shapes(H, G, tiled):
    M, dev = 150, torch.device("cuda:0")
    w = synth.moe_weights(E, H, I, G, seed=86, device=dev)
    ew = (w.gate_up_packed, w.gate_up_scale, w.down_packed, w.down_scale)
    tiles = _lib.tile_experts(*ew, G) if tiled else None
    idx, n = _routing(M, 20, 82)
    assert n == 148
    idx = idx.to(dev)
    wt = torch.rand(M, K, generator=torch.Generator().manual_seed(83)).to(dev)
    x = synth.activations(M, H, seed=84, device=dev)
    y = _lib.moe_forward(x, idx, wt, *ew, G, tiles=tiles)
    for m in range(0, M, 32):
        s = slice(m, m + 32)
        assert torch.equal(_lib.moe_forward(x[s], idx[s], wt[s], *ew, G, tiles=tiles), y[s]), f"rows {m}.."


@pytest.mark.parametrize("M,n_full,slots", [(112, 0, 128), (112, 1, 129), (121, 20, 148), (128, 42, 170),
                                            (128, 43, 171)])
@pytest.mark.parametrize("G,tiled", [(128, False), (128, True), (32, True)])
def test_two_rounds_own_plan(M, n_full, slots, G, tiled):
    # the launch plans for itself (896 <= M * top_k <= 1024); the router's rows make it choose this routing
    dev = torch.device("cuda:0")
    w = synth.moe_weights(E, H, I, G, seed=91, device=dev)
    ew = (w.gate_up_packed, w.gate_up_scale, w.down_packed, w.down_scale)
    tiles = _lib.tile_experts(*ew, G) if tiled else None
    want, n = _routing(M, n_full, 92)
    assert n == slots
    # expert e's router weights are coordinate e, a row's coordinates its experts' scores, best first
    proj = torch.zeros(E, H, dtype=torch.bfloat16)
    proj[torch.arange(E), torch.arange(E)] = 1.0
    rows = torch.zeros(M, H).scatter_(1, want, torch.linspace(8.0, 4.5, K).expand(M, K).contiguous())
    x = synth.activations(M, H, seed=93, device=dev)
    one = torch.ones(H, dtype=torch.bfloat16, device=dev)
    pes = torch.ones(E, dtype=torch.bfloat16, device=dev)
    print(f"own plan M={M} slots={slots} tiled={tiled}", flush=True)
    out, wt, idx = _lib.moe_layer_forward(rows.to(torch.bfloat16).to(dev), one, 1.0, proj.to(dev), pes, 1e-6, K, x,
                                          *ew, G, tiles=tiles)
    assert torch.equal(idx.cpu(), want)
    for m in range(0, M, 32):
        s = slice(m, m + 32)
        assert torch.equal(_lib.moe_forward(x[s], idx[s], wt[s], *ew, G, tiles=tiles), out[s]), f"rows {m}.."
