"""Host views that every launcher takes (ltx_amd/_lib.py): ``row_view`` against
the rule it implements, over 1- to 3-D strided forms, and ``flat``."""

from __future__ import annotations

import pytest
import torch

from ltx_amd import _lib


def _uniform(t):
    """Row stride when the leading dims collapse to one stride, else None."""
    if t.stride(-1) != 1:
        return None
    expect = row = t.stride(-2)
    for size, stride in zip(reversed(t.shape[:-1]), reversed(t.stride()[:-1])):
        if size != 1:
            if stride != expect:
                return None
            expect = stride * size
    return row


BASE = torch.arange(4 * 6 * 32, dtype=torch.float32)


@pytest.mark.parametrize("shape,stride", [
    ((6, 32), (32, 1)), ((6, 16), (32, 1)), ((1, 16), (40, 1)), ((6, 16), (1, 6)), ((0, 16), (32, 1)),
    ((1, 6, 32), (192, 32, 1)), ((1, 6, 16), (7, 32, 1)), ((1, 1, 16), (5, 3, 1)), ((1, 6, 8), (192, 32, 2)),
    ((4, 6, 32), (192, 32, 1)), ((4, 6, 16), (192, 32, 1)), ((4, 3, 16), (192, 32, 1)), ((4, 1, 16), (192, 9, 1)),
])
def test_row_view(shape, stride):
    t = BASE.as_strided(shape, stride)
    v, rs = _lib.row_view(t, shape[-1])
    want = _uniform(t)
    if want is None:  # copied to dense rows
        assert v.is_contiguous() and rs == shape[-1]
    else:
        assert v.data_ptr() == t.data_ptr() and rs == want
    assert torch.equal(v, t)


def test_row_view_refuses_other_widths():
    with pytest.raises(ValueError):
        _lib.row_view(BASE.view(24, 32), 16)


def test_flat():
    dense, strided = BASE[:32].view(1, 1, 32), BASE.view(24, 32)[:, 3]
    assert _lib.flat(dense) is dense
    f = _lib.flat(strided)
    assert f.is_contiguous() and torch.equal(f, strided)


def test_stream_of_refuses_host_tensors():
    with pytest.raises(ValueError):
        _lib.stream_of(BASE)
