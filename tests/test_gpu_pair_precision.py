"""The probabilities keep their 32 bits in the PV product: with P and the
denominator exact, what is left against 64 bits is fp32 sums and exp2 (some
1e-6 relative).  P rounded once to F16 is off by up to 2^-12 of each weight,
2^-12 / sqrt(3) = 1.4e-4 rms over the output, whatever the split."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_parity import _rand_case, mx, run_gpu  # noqa: F401

pytestmark = pytest.mark.gpu

BOUND = 2e-5   # bf16 pairs carry 2^-17 of each weight: 4.4e-6 rms


@pytest.mark.parametrize("kv_type,Sq,Skv,mask,B,Nh,Nkv", [
    # the register decode kernel: Q8_0 with every mask form, odd rows
    (8, 1, 700, None, 1, 32, 8),
    (8, 1, 4096, "causal", 1, 32, 8),
    (8, 1, 4095, "random", 2, 8, 2),
    (8, 5, 2048, "random", 4, 8, 2),
    (1, 1, 4095, "random", 1, 32, 8),
    (1, 1, 701, "random", 1, 32, 8),
    (30, 1, 4095, "random", 1, 32, 8),
    # the LDS decode kernel
    (1, 1, 412, "random", 1, 16, 8),
    (1, 1, 4096, "random", 2, 32, 8),
    (1, 7, 2048, None, 1, 32, 8),
    (30, 1, 4096, "random", 2, 32, 8),
    # prefills under odd rows
    (1, 100, 301, "random", 2, 16, 4),
    (1, 300, 333, "causal", 2, 64, 8),
    (1, 70, 1701, "random", 2, 8, 2),
    (30, 100, 301, "random", 2, 16, 4),
])
def test_probabilities_keep_their_bits(mx, kv_type, Sq, Skv, mask, B, Nh, Nkv):  # noqa: F811
    import oracle

    c = _rand_case(300 + Sq + Skv, kv_type=kv_type, B=B, Sq=Sq, Nh=Nh, Nkv=Nkv, Skv=Skv, mask=mask)
    if kv_type == 8:   # V of scale 2^-6: its values are exact in F16, so that P's bits alone show
        c.v.buf = c.v.buf.copy()
        c.v.buf.view(np.uint8).reshape(-1, 34)[:, :2] = (0x00, 0x24)
    ref = oracle.fa_exact(c.q, c.k, c.v, c.mask, c.scale, 0.0, 0.0, q_round=True).astype(np.float64)
    err = np.linalg.norm(run_gpu(mx, c) - ref) / np.linalg.norm(ref)
    print(f"type {kv_type} {Sq}x{Skv} {mask}: {err:.2e}", flush=True)
    assert err < BOUND
