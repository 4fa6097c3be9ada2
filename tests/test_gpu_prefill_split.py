"""Key-split prefill (few query tiles over many keys): the tiles of a job dealt
to 2..16 workgroups and merged, at the bar of test_gpu_parity.py; the same bits
on every run, for both forms of a mask, and a call that cannot get a workspace."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_graph import no_gc
from test_gpu_parity import _rand_case, check, mx, run_gpu  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Sq,Skv,mask,kw", [
    (64, 24 * 64, None, {}),                          # 3 parts of 8 tiles
    (65, 25 * 64 + 1, None, dict(kv_type=30)),        # a last tile of one key
    (64, 132 * 64, None, dict(Nh=2, Nkv=1)),          # 16 parts of 9 tiles (the last ones shorter)
    (130, 31 * 64, "causal", dict(B=2)),
    (300, 1700, "causal", dict(Nh=16, Nkv=4)),        # 48 jobs
    (200, 1601, "random", dict(mask_heads=2)),        # odd rows, finite values
    (256, 1600, "band", dict(max_bias=4.0)),          # rows of few tiles: fewer parts, some none
    (100, 2048, "random", dict(kv_type=30, Nh=4, Nkv=4)),
    (100, 1344, "causal", dict(kv_type=8)),           # Q8_0, 21 tiles
    (64, 1280, None, dict(kv_type=8)),
])
def test_split_shapes(mx, Sq, Skv, mask, kw):  # noqa: F811
    c = _rand_case(1000 + Sq + Skv, **{"B": 1, "Sq": Sq, "Skv": Skv, "mask": mask, "Nh": 8, "Nkv": 2, **kw})
    got, _ = check(mx, c, f"key split {Sq} x {Skv} {mask} {kw}")
    for _ in range(3):
        assert np.array_equal(run_gpu(mx, c), got)


@pytest.mark.parametrize("spec", [dict(causal=True, pos0=1500), dict(causal=True, pos0=20), dict(lengths=[0, 1700]),
                                  dict(window=300, pos0=600), dict(lengths=[1000, 1601], causal=True, pos0=1000)])
@pytest.mark.parametrize("Skv", [1601, 1700])
def test_split_structured_equals_dense(mx, spec, Skv):  # noqa: F811
    import torch

    from mxfa import cases

    c = _rand_case(1060 + Skv, B=2, Sq=150, Nh=8, Nkv=2, Skv=Skv, mask=None)
    dense = run_gpu(mx, cases.with_dense_mask(c, spec))
    q, k, v = (mx.upload(t) for t in (c.q, c.k, c.v))
    out = mx.flash_attn_ext_masked(q, k, v, mx.mask_spec(**spec), c.scale)
    torch.cuda.synchronize()
    got = mx.output_tensor(out).cpu().numpy()
    if Skv % 4:   # odd mask rows carry P as a hi/lo pair; the spec's weights are off by at most 2^-11 of themselves
        assert np.abs(got - dense).max() <= 2.1 * 2.0 ** -11 * np.abs(c.v.buf.view(np.float16)).max()
    else:
        assert np.array_equal(got, dense)


def test_split_fully_masked_rows(mx):  # noqa: F811
    c = _rand_case(1080, B=1, Sq=140, Nh=4, Nkv=2, Skv=1600, mask="random")
    bits = c.mask.buf.reshape(140, 1600).copy()
    bits[3] = bits[128:] = 0xFC00                     # a row, and a whole query tile
    c.mask.buf = bits.reshape(-1)
    got, _ = check(mx, c, "key split, dead rows")
    assert np.all(got[0, 3] == 0.0) and np.all(got[0, 128:] == 0.0)


def test_split_capture_without_workspace(mx):  # noqa: F811
    """A structured prefill needs no workspace unsplit, and was captured
    without one: it still is, unsplit.  A stream that has one replays the
    split call bit for bit."""
    import torch

    c = _rand_case(1090, B=1, Sq=96, Nh=4, Nkv=2, Skv=2000, mask=None)
    q, k, v = (mx.upload(t) for t in (c.q, c.k, c.v))
    spec = mx.mask_spec(causal=True, pos0=1800)
    ref = mx.output_tensor(mx.flash_attn_ext_masked(q, k, v, spec, c.scale)).clone()
    out = mx.flash_attn_ext_masked(q, k, v, spec, c.scale)
    for warm in (False, True):
        torch.cuda.synchronize()
        mx.release()   # (streams come from a pool: an earlier test may have warmed this one)
        side = torch.cuda.Stream()
        if warm:
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                mx.flash_attn_ext_masked(q, k, v, spec, c.scale, dst=out)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with no_gc(), torch.cuda.graph(g, stream=side):
            mx.flash_attn_ext_masked(q, k, v, spec, c.scale, dst=out)
        assert (mx.workspace_info()[0] > 0) == warm
        for _ in range(3):
            out.owner.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert (out.owner - ref).abs().max().item() <= 2e-3
            assert torch.equal(out.owner, ref) == warm
