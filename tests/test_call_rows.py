"""The calls take their rows in any shape that holds them: a second operand (a
residual delta, the router's input, the attention output) whose matrix has
another width than the first's rows is read as rows of that width."""
import pytest
import torch

from hybridagent_amd import _lib, synth


@pytest.mark.parametrize("shape", [(6, 8), (3, 16), (12, 4), (48,), (2, 3, 8), (1, 48), (6, 1, 8)])
def test_rows_of_any_shape(shape):
    t = torch.arange(48.0).reshape(shape)
    r = _lib._rows(t, 8)
    assert r.shape == (6, 8) and torch.equal(r, torch.arange(48.0).reshape(6, 8))


def test_rows_that_do_not_fit_are_refused():
    with pytest.raises(RuntimeError):
        _lib._rows(torch.zeros(3, 7), 8)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(2, 512), (8, 128), (1, 1024), (4, 1, 256)])
def test_add_rms_norm_delta_of_another_width(shape):
    dev = torch.device("cuda:0")
    h = synth.activations(4, 256, seed=1, device=dev)
    d = synth.activations(4, 256, seed=2, device=dev)
    w = torch.ones(256, dtype=torch.bfloat16, device=dev)
    x, y = _lib.add_rms_norm(h, w, 1e-6, d.reshape(shape))
    x0, y0 = _lib.add_rms_norm(h, w, 1e-6, d)
    assert torch.equal(x, x0) and torch.equal(y, y0)
