"""Calls repeated back to back: every run right (at the bar of
test_gpu_parity.py) and the same bits, on every prefill kernel over 1 to 6 key
tiles, whatever the instruction cache holds."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_parity import _rand_case, check, mx  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kv_type", [1, 30])
@pytest.mark.parametrize("mask", [None, "zeros", "random"])
@pytest.mark.parametrize("Skv", [64, 128, 192, 237, 240, 256, 300, 384])
@pytest.mark.parametrize("Sq,Nh", [(100, 8), (129, 64)])      # 64-query workgroups; 128 and 192
def test_repeated_calls(mx, Sq, Nh, Skv, mask, kv_type):  # noqa: F811
    import torch

    c = _rand_case(1200 + Sq + Skv, B=2, Sq=Sq, Nh=Nh, Nkv=Nh // 8, Skv=Skv, mask=mask and "random", kv_type=kv_type)
    if mask == "zeros":   # padding: the last 33 keys
        bits = c.mask.buf.reshape(-1, Skv).copy()
        bits[:] = 0
        bits[:, Skv - 33:] = 0xFC00
        c.mask.buf = bits.reshape(-1)
    want, _ = check(mx, c, f"repeat {Sq} x {Skv} {mask} t{kv_type}", strict=False)
    q, k, v = (mx.upload(t) for t in (c.q, c.k, c.v))
    m = mx.upload(c.mask) if c.mask is not None else None
    out = mx.flash_attn_ext(q, k, v, m, c.scale)
    runs = []
    for _ in range(6):
        out.owner.fill_(float("nan"))
        mx.flash_attn_ext(q, k, v, m, c.scale, dst=out)
        runs.append(mx.output_tensor(out).clone())
    torch.cuda.synchronize()
    for r in runs:
        assert np.array_equal(r.cpu().numpy(), want)
