"""The grids on both sides of the rule for the 192-query prefill kernel
(fa_wide.hip): one workgroup per CU, two per CU of the 128-query kernel; and a
dense mask against its structured form there, bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_parity import _rand_case, check, mx, run_gpu  # noqa: F401

pytestmark = pytest.mark.gpu


# 128 heads, unmasked: 2 x 128 192-query workgroups (257 queries), 3 x 128 of
# them and 4 x 128 128-query ones (385), 5 x 128 of the latter (513).
@pytest.mark.parametrize("Sq", [257, 385, 513])
@pytest.mark.parametrize("Skv,mask", [(63, None), (321, None), (240, "random")])
def test_wide_rule(mx, Sq, Skv, mask):  # noqa: F811
    c = _rand_case(900 + Sq + Skv, B=1, Sq=Sq, Skv=Skv, mask=mask, Nh=128, Nkv=8)
    check(mx, c, f"128 heads, {Sq} x {Skv} {mask}")


@pytest.mark.parametrize("Sq", [385, 513])
@pytest.mark.parametrize("spec", [dict(causal=True, pos0=70), dict(lengths=[130])])
def test_wide_rule_structured_equals_dense(mx, Sq, spec):  # noqa: F811
    import torch

    from mxfa import cases

    c = _rand_case(950 + Sq, B=1, Sq=Sq, Nh=128, Nkv=8, Skv=240, mask=None)
    dense = run_gpu(mx, cases.with_dense_mask(c, spec))
    q, k, v = (mx.upload(t) for t in (c.q, c.k, c.v))
    out = mx.flash_attn_ext_masked(q, k, v, mx.mask_spec(**spec), c.scale)
    torch.cuda.synchronize()
    assert np.array_equal(mx.output_tensor(out).cpu().numpy(), dense)
