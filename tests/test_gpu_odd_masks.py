"""Prefill under dense masks whose rows are not 8-byte aligned: the [S, S]
masks of the DiT (src/dit-sampler.h:262-309) and the encoders
(src/qwen3-enc.h:429-437) for every S that is not a multiple of 4.  They run
the MFMA prefill kernel (2-byte aligned classifier loads, the last group of a
row shifted into place), at the bar of test_gpu_parity.py."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_graph import no_gc
from test_gpu_parity import _rand_case, check, mx, run_gpu  # noqa: F401

pytestmark = pytest.mark.gpu


def _repitch(mask, extra, shift):
    """The mask with `extra` entries between rows and `shift` before the
    first; the gaps hold NaN, which no load may let through."""
    from mxfa.cases import HostView

    Skv, Sq, Hm, B = mask.ne
    pitch = Skv + extra
    buf = np.full(B * Hm * Sq * pitch + shift, 0x7E00, dtype=np.uint16)
    dst = buf[shift:].reshape(B, Hm, Sq, pitch)
    dst[..., :Skv] = mask.buf.view(np.uint16).reshape(B, Hm, Sq, Skv)
    return HostView(1, (Skv, Sq, Hm, B), (2, 2 * pitch, 2 * pitch * Sq, 2 * pitch * Sq * Hm), buf, offset=2 * shift)


def _kernels(mx_, call):
    import torch

    mx_.timing_reset()
    mx_.timing_enable(1)
    call()
    torch.cuda.synchronize()
    mx_.timing_enable(0)
    n = {f: mx_.timing_read(f)[1] for f in ("fa_prefill", "fa_decode", "mask_classify")}
    mx_.timing_reset()
    return n


# (edges of the 128 x 64 tiles, every remainder of 4 keys, short rows)
@pytest.mark.parametrize("Sq,Skv,mask,kw,extra,shift", [
    (64, 5, "random", {}, 0, 0),
    (65, 63, "random", dict(Nkv=8), 0, 1),
    (127, 129, "causal", {}, 0, 0),
    (129, 255, "band", dict(mask_heads=2), 0, 3),
    (130, 258, "random", dict(mask_heads=8, kv_type=30), 0, 0),
    (257, 257, "causal", dict(kv_type=30), 0, 0),
    (200, 323, "random", dict(softcap=20.0, max_bias=8.0), 0, 0),
    (300, 301, "band", dict(max_bias=4.0), 3, 2),
    (96, 322, "band", {}, 0, 0),
    (70, 4, "random", {}, 1, 1),
])
def test_odd_mask_rows(mx, Sq, Skv, mask, kw, extra, shift):  # noqa: F811
    c = _rand_case(700 + Sq + Skv, B=2, Sq=Sq, Skv=Skv, mask=mask, **{"Nh": 8, "Nkv": 2, **kw})
    c.mask = _repitch(c.mask, extra, shift)
    n = _kernels(mx, lambda: run_gpu(mx, c))
    assert n["fa_prefill"] == 1 and n["fa_decode"] == 0, n
    check(mx, c, f"odd mask rows {Sq} x {Skv} {mask} {kw} +{extra} @{shift}")


def test_odd_rows_equal_padded_rows(mx):  # noqa: F811
    """The same mask in odd rows (P as a hi/lo pair) and in rows padded to 8
    bytes (weights off by at most 2^-11 of themselves: 2 * 2^-11 * max|V|)."""
    c = _rand_case(751, B=2, Sq=261, Nh=8, Nkv=2, Skv=337, mask="random")
    odd = run_gpu(mx, c)
    c.mask = _repitch(c.mask, 3, 0)
    c.mask.ne = (340,) + tuple(c.mask.ne[1:])   # rows of 340 entries, 8-byte aligned
    bound = 2.1 * 2.0 ** -11 * np.abs(c.v.buf.view(np.float16)).max()
    assert np.abs(odd - run_gpu(mx, c)).max() <= bound


def test_odd_rows_under_capture_without_reserve(mx):  # noqa: F811
    """A captured call whose workspace cannot hold the mask's classes keeps to
    the decode kernel, as it did before odd rows reached the prefill kernel
    (here 1088 streams of 16 rows: one split, no partials)."""
    import torch

    c = _rand_case(752, B=2, Sq=65, Nh=128, Nkv=32, Skv=69, mask="random")
    q, k, v, m = (mx.upload(t) for t in (c.q, c.k, c.v, c.mask))
    ref = mx.output_tensor(mx.flash_attn_ext(q, k, v, m, c.scale)).clone()
    out = mx.flash_attn_ext(q, k, v, m, c.scale)
    torch.cuda.synchronize()
    mx.release()   # (streams come from a pool: an earlier test may have warmed this one)
    side = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    with no_gc(), torch.cuda.graph(g, stream=side):
        mx.graph_begin()
        mx.flash_attn_ext(q, k, v, m, c.scale, dst=out)
        mx.graph_end()
    assert mx.workspace_info()[0] == 0
    for _ in range(3):
        out.owner.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert (out.owner - ref).abs().max().item() <= 2e-3
        assert not torch.equal(out.owner, ref)   # the prefill kernel's bits are others
