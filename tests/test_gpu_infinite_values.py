"""An infinity in V of a key that every query sees is one in the output, of the
same sign, and touches no other value: in F16, where P goes into the PV
product as a pair whose parts are both positive, and in the splits' merge,
whose slots past the last split are not added."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_parity import _rand_case, mx, run_gpu  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Sq,Skv,Nh,mask", [
    # the LDS decode kernel: one key (P = 1), one split, several, 9 of 16 merge slots
    (1, 1, 2, None), (1, 64, 8, None), (1, 412, 16, "zeros"), (5, 580, 8, "zeros"), (1, 4096, 8, None),
    # the register kernel (odd mask rows)
    (1, 1, 2, "zeros"), (1, 411, 16, "zeros"), (7, 2047, 8, "zeros"),
    # prefills under odd rows: fa_narrow.hip, key split, fa_mfma.hip
    (100, 238, 16, "zeros"), (70, 70, 8, "causal"), (128, 1701, 8, "zeros"), (300, 333, 64, "zeros"),
])
def test_infinite_values(mx, Sq, Skv, Nh, mask):  # noqa: F811
    c = _rand_case(500 + Sq + Skv, B=2, Sq=Sq, Nh=Nh, Nkv=2, Skv=Skv, mask=mask and "causal")
    if mask == "zeros":
        c.mask.buf = np.zeros_like(c.mask.buf)
    clean = run_gpu(mx, c)
    c.v.buf = c.v.buf.copy()
    v = c.v.buf.reshape(2, 2, Skv, 128)
    v[:, :, 0, 7] = 0x7C00          # key 0: the first split
    v[:, :, 0, 9] = 0xFC00
    last = Skv - 1 if mask != "causal" else 0
    v[:, :, last, 11] = 0x7C00      # the last split
    got = run_gpu(mx, c)
    assert np.isposinf(got[..., 7]).all() and np.isneginf(got[..., 9]).all() and np.isposinf(got[..., 11]).all()
    rest = np.setdiff1d(np.arange(128), [7, 9, 11])
    assert np.array_equal(got[..., rest], clean[..., rest])
