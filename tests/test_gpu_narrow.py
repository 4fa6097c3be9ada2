"""The 64-query prefill kernel (fa_narrow.hip) at the edges of its tiles and
of the grids it serves, at the bar of test_gpu_parity.py; and the two forms of
a mask bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_parity import _rand_case, check, mx, run_gpu  # noqa: F401

pytestmark = pytest.mark.gpu


# Grids of at most 256 workgroups run four stages, unmasked ones of 257..512
# two; key counts around the ring (1..5 tiles of 64) and a partial last tile.
@pytest.mark.parametrize("Sq,Skv,mask,kw", [
    (64, 64, None, {}),
    (65, 1, None, dict(kv_type=30)),
    (127, 129, None, dict(Nh=32, Nkv=8)),          # 128 workgroups
    (129, 193, None, dict(Nh=128, Nkv=8)),         # 768: past the rule
    (129, 321, None, dict(Nh=64, Nkv=8)),          # 384: two stages
    (65, 257, None, dict(Nh=64, Nkv=8, kv_type=30)),
    (100, 320, None, dict(softcap=15.0)),
    (200, 384, "causal", {}),
    (200, 1000, "causal", dict(kv_type=30)),
    (191, 324, "random", dict(mask_heads=2)),
    (300, 300, "band", dict(max_bias=8.0)),
    (72, 128, "random", dict(softcap=30.0, kv_type=30, mask_heads=8)),
])
def test_narrow_shapes(mx, Sq, Skv, mask, kw):  # noqa: F811
    c = _rand_case(800 + Sq + Skv, B=2, Sq=Sq, Skv=Skv, mask=mask, **{"Nh": 8, "Nkv": 2, **kw})
    check(mx, c, f"64-query kernel {Sq} x {Skv} {mask} {kw}")


@pytest.mark.parametrize("spec", [
    dict(causal=True, pos0=70), dict(window=40), dict(causal=True, window=90, pos0=3),
    dict(lengths=[0, 130]), dict(lengths=[257, 64], causal=True),
])
@pytest.mark.parametrize("Skv", [257, 260])
def test_narrow_structured_equals_dense(mx, spec, Skv):  # noqa: F811
    import torch

    from mxfa import cases

    c = _rand_case(860 + Skv, B=2, Sq=150, Nh=8, Nkv=2, Skv=Skv, mask=None)
    dense = run_gpu(mx, cases.with_dense_mask(c, spec))
    q, k, v = (mx.upload(t) for t in (c.q, c.k, c.v))
    out = mx.flash_attn_ext_masked(q, k, v, mx.mask_spec(**spec), c.scale)
    torch.cuda.synchronize()
    got = mx.output_tensor(out).cpu().numpy()
    if Skv % 4:   # odd mask rows carry P as a hi/lo pair; the spec's weights are off by at most 2^-11 of themselves
        assert np.abs(got - dense).max() <= 2.1 * 2.0 ** -11 * np.abs(c.v.buf.view(np.float16)).max()
    else:
        assert np.array_equal(got, dense)


def test_narrow_fully_masked_rows_and_tiles(mx):  # noqa: F811
    """Rows, 64-query halves and key tiles with no live key; NaN in K / V that
    no row may see."""
    c = _rand_case(880, B=1, Sq=192, Nh=4, Nkv=4, Skv=256, mask="causal")
    bits = c.mask.buf.reshape(1, 1, 192, 256).copy()
    bits[0, 0, 5] = bits[0, 0, 64:128] = 0xFC00
    bits[0, 0, :, 64:128] = 0xFC00
    c.mask.buf = bits.reshape(-1)
    for t in (c.k, c.v):
        t.buf = t.buf.copy()
        t.buf.reshape(4, 256, 128)[:, 64:128] = 0x7E00
    got = run_gpu(mx, c)
    assert np.all(got[0, 5] == 0.0) and np.all(got[0, 64:128] == 0.0) and not np.isnan(got).any()
    c2 = _rand_case(880, B=1, Sq=192, Nh=4, Nkv=4, Skv=256, mask="causal")
    c2.mask.buf = bits.reshape(-1)
    assert np.array_equal(got, run_gpu(mx, c2))
