"""Linear4Bit at prefill sizes (k_linear_w4): every tile height and its edges, odd
widths, a last half k stage (K % 64 == 32), odd group counts, group sizes whose
last group is partial, a bias, an input with infinities and NaN in single rows.

Reference: the float64 product of the bf16 inputs and bf16_RNE(q * s) weights.
A fp32 sum of K products in any order is off by at most K 2^-24 of the sum of
their magnitudes; the result rounds to bf16 (7 stored mantissa bits) once: at
most half a unit, 2^-8 of the value."""
import pytest
import torch

from hybridagent_amd import _lib, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    assert _lib.available(), "libw4a16moe.so must be built"
    return torch.device("cuda:0")


def _weights(N, K, G, seed, dev):
    p = synth.packed_int4((N, K), seed, dev)
    s = synth.group_scales((N, K), G, seed + 1, dev)
    sh = torch.arange(0, 32, 4, dtype=torch.int32, device=dev)
    q = (((p.unsqueeze(-1) >> sh) & 15) - 8).reshape(N, K).float()
    w = (q * s.float().repeat_interleave(G, 1)[:, :K]).to(torch.bfloat16).double()
    return p, s, w


def _check(y, x, w, b, K, what):
    ref = x.double() @ w.t()
    mag = x.double().abs() @ w.abs().t()
    if b is not None:
        ref, mag = ref + b.double(), mag + b.double().abs()
    bound = 2.0 ** -8 * ref.abs() + (1 + 2.0 ** -8) * (K + 1) * 2.0 ** -24 * mag
    bad = (y.double() - ref).abs() > bound
    assert not bad.any(), f"{what}: {int(bad.sum())} of {bad.numel()}"


# the tiled GEMM takes more than 900e3 outputs.  N: one column tile and less, tiles' edges, odd; K: whole and partial
# last tiles; rows past whole tiles; 228 groups (scales fill LDS), 232 and a partial tile past K = 3072 (streamed)
@pytest.mark.parametrize("M,K,N,G", [(481, 160, 2816, 32), (1001, 160, 2816, 32), (512, 704, 2816, 128),
                                     (700, 2144, 1357, 32), (330, 2816, 2816, 32), (3600, 1056, 257, 64),
                                     (3601, 352, 256, 32), (481, 2080, 2111, 128), (65, 224, 14000, 32),
                                     (330, 9216, 2816, 128), (330, 7296, 2816, 32), (330, 7424, 2816, 32),
                                     (330, 3232, 2816, 32)])
def test_linear_prefill_shapes(dev, M, K, N, G):
    p, s, w = _weights(N, K, G, 51, dev)
    x = synth.activations(M, K, 53, dev)
    b = synth.activations(1, N, 54, dev)[0] if N % 2 else None
    _check(_lib.linear(x, p, s, b, G), x, w, b, K, f"M={M} K={K} N={N} G={G}")


# every tile height: one round of 1 .. 6 blocks at these rows, then two rounds
@pytest.mark.parametrize("M", [600, 800, 1200, 1700, 2048, 2300, 3000, 4096, 5000])
def test_linear_prefill_rows(dev, M):
    K, N, G = 704, 2816, 32
    p, s, w = _weights(N, K, G, 61, dev)
    x = synth.activations(M, K, 63, dev)
    _check(_lib.linear(x, p, s, None, G), x, w, None, K, f"M={M}")


def test_linear_prefill_nonfinite_rows_stay_apart(dev):
    # K % 64 == 32: the lanes without k in the last stage hold other bytes of the row, which must not count
    M, K, N, G = 512, 2144, 2816, 32
    p, s, w = _weights(N, K, G, 71, dev)
    x = synth.activations(M, K, 73, dev)
    clean = _lib.linear(x, p, s, None, G)
    y = x.clone()
    y[3, 2112] = float("inf")   # in the last stage: 32 k of it
    y[7, 5] = float("nan")
    got = _lib.linear(y, p, s, None, G)
    keep = torch.ones(M, dtype=torch.bool, device=dev)
    keep[3] = keep[7] = False
    assert torch.equal(got[keep], clean[keep])
    assert got[7].isnan().all()
    col = w[:, 2112]
    assert torch.equal(got[3] == float("inf"), col > 0)
    assert torch.equal(got[3] == float("-inf"), col < 0)
    assert got[3][col == 0].isnan().all()
