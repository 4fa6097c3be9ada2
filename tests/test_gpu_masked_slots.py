"""NaN and infinities in K and V of keys that no query may see change no bit of
a prefill: such keys end inside a tile, at the end (padding, an unwritten
cache) or in front, under odd and aligned dense masks and their structured
form, on every prefill kernel and in its key-split form."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_parity import _rand_case, check, mx, run_gpu  # noqa: F401

pytestmark = pytest.mark.gpu


def _poison(c, dead):
    if c.k.type == 8:   # a NaN scale in every block
        for t in (c.k, c.v):
            t.buf = t.buf.copy()
            t.buf.view(np.uint8).reshape(-1, t.ne[1], 4, 34)[:, dead, :, :2] = (0x00, 0x7E)
        return
    nan, inf = (0x7E00, 0x7C00) if c.k.type == 1 else (0x7FC0, 0x7F80)
    for t, even, odd in ((c.k, nan, inf), (c.v, inf, nan)):
        t.buf = t.buf.copy()
        rows = t.buf.reshape(-1, t.ne[1], 128)
        rows[:, dead[::2]] = even
        rows[:, dead[1::2]] = odd


@pytest.mark.parametrize("kv_type", [1, 30, 8])
@pytest.mark.parametrize("Sq,Skv,live,mask,kw", [
    # fa_narrow.hip: odd and aligned rows, finite values, a mask per head
    (100, 238, (0, 207), "zeros", {}),
    (100, 240, (0, 207), "zeros", {}),
    (192, 257, (0, 129), "random", {}),
    (150, 301, (37, 290), "zeros", dict(mask_heads=2)),
    # fa_mfma.hip, and fa_wide.hip for F16 over at most 4 aligned key tiles
    (129, 238, (0, 207), "zeros", dict(Nh=64, Nkv=8)),
    (129, 240, (3, 207), "zeros", dict(Nh=64, Nkv=8)),
    (400, 256, (17, 193), "random", dict(Nh=64, Nkv=8, B=1)),
    (129, 333, (70, 331), "random", dict(Nh=64, Nkv=8)),
    (385, 512, (0, 461), "zeros", dict(Nh=64, Nkv=8, B=1)),
    # key split, and rows of more than 64 key tiles
    (128, 1701, (3, 1630), "zeros", {}),
    (128, 1700, (0, 1699), "random", dict(B=1)),
    (64, 4500, (0, 4201), "zeros", dict(B=1, Nh=2, Nkv=1)),
    (65, 4501, (100, 4201), "zeros", dict(B=4, Nh=32, Nkv=1)),
])
def test_non_finite_dead_keys(mx, Sq, Skv, live, mask, kw, kv_type):  # noqa: F811
    c = _rand_case(760 + Sq + Skv, kv_type=kv_type, Sq=Sq, Skv=Skv, mask="random",
                   **{"B": 2, "Nh": 8, "Nkv": 2, **kw})
    bits = c.mask.buf.reshape(-1, Skv).copy()
    if mask == "zeros":
        bits[:] = 0
    bits[:, :live[0]] = bits[:, live[1]:] = 0xFC00
    c.mask.buf = bits.reshape(-1)
    clean = run_gpu(mx, c)
    assert np.isfinite(clean).all()
    _poison(c, np.r_[0:live[0], live[1]:Skv])
    assert np.array_equal(run_gpu(mx, c), clean)


@pytest.mark.parametrize("Sq,Skv,spec,kw", [
    (100, 238, dict(lengths=[207, 207]), {}),
    (150, 400, dict(window=40, pos0=150), {}),                        # keys 110 .. 339
    (129, 240, dict(lengths=[207]), dict(Nh=64, Nkv=8)),
    (385, 700, dict(window=30, pos0=100), dict(Nh=64, Nkv=8, B=1)),   # 70 .. 514
    (300, 700, dict(causal=True, pos0=250), dict(Nh=64, Nkv=8, B=1)),
    (128, 1701, dict(causal=True, pos0=1500), dict(B=1)),
])
def test_non_finite_outside_the_spec(mx, Sq, Skv, spec, kw):  # noqa: F811
    import torch

    c = _rand_case(800 + Sq + Skv, Sq=Sq, Skv=Skv, mask=None, **{"B": 2, "Nh": 8, "Nkv": 2, **kw})
    i, j, p = np.arange(Sq)[:, None], np.arange(Skv)[None, :], spec.get("pos0", 0)
    live = (j < spec.get("lengths", [Skv])[0]) & (np.abs(p + i - j) <= spec.get("window", Skv + Sq + p))
    if spec.get("causal"):
        live &= j <= p + i

    def run():
        q, k, v = (mx.upload(t) for t in (c.q, c.k, c.v))
        out = mx.flash_attn_ext_masked(q, k, v, mx.mask_spec(**spec), c.scale)
        torch.cuda.synchronize()
        return mx.output_tensor(out).cpu().numpy()

    clean = run()
    _poison(c, np.flatnonzero(~live.any(axis=0)))
    got = run()
    assert np.isfinite(clean).all() and np.array_equal(got, clean)


def test_per_sequence_padding(mx):  # noqa: F811
    """Sequences of different lengths: what is padding in one is live in the
    other."""
    c = _rand_case(840, B=2, Sq=140, Nh=8, Nkv=2, Skv=246, mask="random")
    bits = c.mask.buf.reshape(2, 140, 246).copy()
    bits[:] = 0
    bits[0, :, 100:] = bits[1, :, 200:] = 0xFC00
    c.mask.buf = bits.reshape(-1)
    clean, _ = check(mx, c, "padded sequences")
    for t in (c.k, c.v):
        t.buf = t.buf.copy()
        rows = t.buf.reshape(2, 2, 246, 128)
        rows[0, :, 100:] = rows[1, :, 200:] = 0x7E00
    assert np.array_equal(run_gpu(mx, c), clean)
