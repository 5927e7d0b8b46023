"""TiledWeights.struct: the C structure follows the fields, and copies and pickles
carry the fields alone."""
import copy
import dataclasses
import pickle

import torch

from hybridagent_amd import _lib


def test_struct_follows_fields_and_copies():
    tw = _lib.TiledWeights(4, 64, 32, 32, gu_decode=torch.zeros(16, dtype=torch.int32))
    a = tw.struct()
    assert (a.E, a.H, a.I, a.group_size) == (4, 64, 32, 32)
    assert (a.gu_decode, a.gu_decode_bytes) == (tw.gu_decode.data_ptr(), 64)
    assert (a.dn_decode, a.dn_decode_bytes) == (None, 0)
    assert tw.struct() is a
    tw.dn_prefill = torch.zeros(8, dtype=torch.int32)
    b = tw.struct()
    assert b is not a and (b.dn_prefill, b.dn_prefill_bytes) == (tw.dn_prefill.data_ptr(), 32)
    assert a.dn_prefill is None, "a structure handed out does not change"
    tw.gu_decode = None
    assert tw.struct().gu_decode is None
    for c in (copy.deepcopy(tw), pickle.loads(pickle.dumps(tw)), copy.copy(tw), dataclasses.replace(tw)):
        assert c.struct().dn_prefill == c.dn_prefill.data_ptr()
        assert torch.equal(c.dn_prefill, tw.dn_prefill)


def test_require_gpu_errors():
    import pytest
    cpu = torch.zeros(1)
    assert _lib._require_gpu(None) is None
    with pytest.raises(RuntimeError, match="GPU only"):
        _lib._require_gpu(None, cpu)
