"""Segment tails of the prefill GEMM: an expert's rows give the same bits whether
they are a tail of one or two 32-row blocks (stages of 128 k with the item's
scales resident, or three column tiles per item on the tiled weights) or part
of a larger segment (stages of 64 k that bring their own scales), at the edges
of the tail classes, with an odd number of 64-wide k blocks, every supported
group size, both weight layouts, and a width whose scales do not fit beside
the ring."""
import numpy as np
import pytest
import torch

import oracle
from checks import margin
from hybridagent_amd import _lib, synth

pytestmark = pytest.mark.gpu

TOL = 1e-2


@pytest.mark.parametrize("tiled", [False, True])
@pytest.mark.parametrize("h,i,G", [(384, 320, 32), (384, 384, 64), (512, 512, 128), (2816, 704, 32), (2816, 704, 128),
                                   (5376, 320, 32)])
def test_tail_rows_bit_identical(h, i, G, tiled):
    dev = torch.device("cuda:0")
    rows = [1, 2, 31, 32, 33, 63, 64, 65, 130]
    e = len(rows)
    wts = synth.moe_weights(e, h, i, G, seed=41, device=dev)
    gpu = [wts.gate_up_packed, wts.gate_up_scale, wts.down_packed, wts.down_scale]
    tiles = _lib.tile_experts(*gpu, G) if tiled else None
    idx = torch.repeat_interleave(torch.arange(e), torch.tensor(rows))
    idx = idx[torch.randperm(idx.numel(), generator=torch.Generator().manual_seed(42))]
    M = idx.numel()
    assert M > 256
    # batch B: 66 tokens more on every expert, so that no segment is a tail of two blocks or fewer
    idx_b = torch.cat([idx, torch.arange(e).repeat(66)])
    x = synth.activations(idx_b.numel(), h, seed=43, device=dev)
    w = torch.ones(idx_b.numel(), 1, device=dev)
    print(f"tails h={h} i={i} G={G} tiled={tiled}", flush=True)
    a = _lib.moe_forward(x[:M], idx[:, None].to(dev), w[:M], *gpu, G, tiles=tiles)
    b = _lib.moe_forward(x, idx_b[:, None].to(dev), w, *gpu, G, tiles=tiles)
    assert torch.equal(a, b[:M])
    pick = torch.cat([(idx == n).nonzero()[:2, 0] for n in range(e)])
    np_ = lambda t: t.float().cpu().numpy()
    bits = lambda t: t.cpu().view(torch.int16).numpy().view(np.uint16)
    ref = oracle.moe_forward(np_(x[pick]), idx[pick][:, None].numpy(), np_(w[pick]), wts.gate_up_packed.cpu().numpy(),
                             bits(wts.gate_up_scale), wts.down_packed.cpu().numpy(), bits(wts.down_scale), G)
    assert margin(f"prefill tails h={h} i={i} G={G}", oracle.max_abs_rel(np_(a[pick]), ref)) <= TOL


@pytest.mark.parametrize("extra", [0, 40])
@pytest.mark.parametrize("h,i,G", [(384, 320, 32), (2816, 704, 128)])
def test_wide_items_only_among_small_tails(h, i, G, extra):
    # every expert a tail of at most 32 rows: the tiled weights' wide items; with one expert of 60 rows: tail items
    dev = torch.device("cuda:0")
    e, r = 18, 20
    wts = synth.moe_weights(e, h, i, G, seed=44, device=dev)
    gpu = [wts.gate_up_packed, wts.gate_up_scale, wts.down_packed, wts.down_scale]
    tiles = _lib.tile_experts(*gpu, G)
    idx = torch.cat([torch.arange(e).repeat(r), torch.zeros(extra, dtype=torch.long)])[:, None].to(dev)
    x = synth.activations(idx.shape[0], h, seed=45, device=dev)
    w = torch.ones(idx.shape[0], 1, device=dev)
    print(f"wide h={h} i={i} G={G} extra={extra}", flush=True)
    a = _lib.moe_forward(x, idx, w, *gpu, G, tiles=tiles)
    assert torch.equal(a, _lib.moe_forward(x, idx, w, *gpu, G, tiles=None))
    if extra:
        assert torch.equal(a[:e * r], _lib.moe_forward(x[:e * r], idx[:e * r], w[:e * r], *gpu, G, tiles=tiles))
