"""Tensor descriptors that ops packs, against the ones _lib.descriptor fills field by field."""
import os
import sys

import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "candle-3d_amd"))

torch = pytest.importorskip("torch")
from lux3d_fused import _lib, ops  # noqa: E402

BASE = torch.zeros(2, 3, 4, 5, 6)


@pytest.mark.parametrize("t", [
    torch.tensor(3.0), torch.zeros(0), torch.zeros(7, dtype=torch.int64), BASE[0, 0, 0].t(),
    BASE.permute(4, 2, 0, 1, 3), BASE[:, 1:, ::2, 3:], BASE[:1, :1, 0, 0, :1].expand(4, 5, 6),
    torch.zeros(0, 8, dtype=torch.bfloat16), torch.zeros(3, 4, dtype=torch.int8)[:, ::2],
], ids=lambda t: f"{t.dtype}-{tuple(t.shape)}-{tuple(t.stride())}")
def test_packed_descriptor_has_the_fields_of_the_tensor(t):
    want = _lib.descriptor(t.data_ptr(), ops._DT[t.dtype], list(t.shape) or [1], list(t.stride()) or [1])
    assert bytes(ops.desc(t).contents) == bytes(want)


def test_descriptor_refusals_and_null():
    assert ops.desc(None) is None
    with pytest.raises(TypeError, match="unsupported dtype"):
        ops.desc(torch.zeros(1, dtype=torch.float64))
    with pytest.raises(IndexError):
        ops.desc(torch.zeros(1, 1, 1, 1, 1, 1))


class _Named(torch.Tensor):
    pass


@pytest.mark.parametrize("x", [BASE.permute(4, 2, 0, 1, 3), BASE[:, :1].expand(2, 3, 4, 5, 6), torch.zeros(()),
                               torch.nn.Parameter(torch.zeros(2, 3)), torch.zeros(2, 3).as_subclass(_Named)],
                         ids=["permuted", "expanded", "scalar", "parameter", "subclass"])
def test_new_outputs_are_contiguous_plain_tensors(x):
    y = ops._new(x)
    assert type(y) is torch.Tensor and y.is_contiguous() and not y.requires_grad
    assert y.shape == x.shape and y.dtype == x.dtype and y.device == x.device
