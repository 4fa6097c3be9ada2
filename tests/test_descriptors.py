"""DeviceView.desc(): the one-call packing and the field-by-field path give the
same descriptor for whatever int() takes, and refuse the same."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")
import mxfa  # noqa: E402


def _by_field(v):
    t = mxfa.MxfaTensor()
    t.type = int(v.type)
    for i in range(4):
        t.ne[i] = int(v.ne[i])
        t.nb[i] = int(v.nb[i])
    t.data = ctypes.c_void_p(int(v.ptr)) if v.ptr else None
    return t


@pytest.mark.parametrize("view", [
    (1, (128, 7, 8, 1), (2, 256, 1792, 14336), 1 << 44),
    (8, [128, 5, 1, 1], [34, 136, 680, 680], 0),
    (0, (128, 3, 2, 1), (4, 512, 1536, 3072), None),
    (np.int32(30), tuple(np.int64(x) for x in (128, 3, 2, 1)), tuple(np.int64(x) for x in (2, 256, 768, 1536)),
     np.uint64(1 << 40)),
    (1.0, (128.0, 3, 2, 1), (2, 256.0, 768, 1536), 4096.0),      # int() takes floats
    (1, (128, -3, 2, 1), (2, -256, 768, 1536), 4096),            # a negative stride wraps, as size_t does
    (1, (128, 3, 2, 1, 9), (2, 256, 768, 1536, 9), 4096),        # the first four
    (1, torch.tensor([128, 3, 2, 1]), torch.tensor([2, 256, 768, 1536]), 4096),
])
def test_desc_matches_fields(view):
    v = mxfa.DeviceView(*view)
    assert bytes(v.desc()) == bytes(_by_field(v))


@pytest.mark.parametrize("view", [(1, (128, 3, 2), (2, 256, 768, 1536), 1), (1, ("a", 3, 2, 1), (2, 256, 768, 1536), 1)])
def test_desc_refuses(view):
    v = mxfa.DeviceView(*view)
    with pytest.raises(Exception) as a:
        _by_field(v)
    with pytest.raises(type(a.value)):
        v.desc()


@pytest.mark.parametrize("ne,nb", [
    ((128, 3, 2, 1, 2), (256, 768, 1536)),           # eight values in all, one on the wrong side
    ((128, 3, 2), (1, 2, 256, 768, 1536)),
])
def test_desc_refuses_a_shifted_split(ne, nb):
    with pytest.raises(IndexError):
        mxfa.DeviceView(1, ne, nb, 4096).desc()
