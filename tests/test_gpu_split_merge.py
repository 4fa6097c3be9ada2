"""The split merge of the decode kernels over the row and split counts where
its work division changes (1, 2 and 4 rows share a row's splits among waves,
others do not; 32 splits are one batch), dead splits among them, at the bar of
test_gpu_parity.py."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_parity import _rand_case, check, mx  # noqa: F401

pytestmark = pytest.mark.gpu

# (test_plan_routes.py holds the split counts: 66 and 130 are odd rows, 1 and 2
# splits of the register kernel, the others 2 to 64 of the LDS kernel)

@pytest.mark.parametrize("Skv", [66, 68, 130, 132, 2048, 2100, 4096, 6000])
@pytest.mark.parametrize("G,Sq", [(1, 1), (2, 1), (3, 1), (4, 1), (1, 7), (8, 2), (3, 6)])
def test_merge_rows_and_splits(mx, G, Sq, Skv):  # noqa: F811
    c = _rand_case(900 + G + Sq + Skv, B=1, Sq=Sq, Nh=G, Nkv=1, Skv=Skv, mask="random")
    live = np.arange(Skv) < Skv - Skv // 3           # the last third of the splits has no live key
    bits = c.mask.buf.reshape(Sq, Skv).copy()
    bits[:, ~live] = 0xFC00
    bits[Sq - 1, 64:128] = 0xFC00                    # a dead split inside the range, for one row
    c.mask.buf = bits.reshape(-1)
    check(mx, c, f"merge G={G} Sq={Sq} Skv={Skv}")


@pytest.mark.parametrize("kv_type,mask", [(8, "random"), (30, None), (8, None)])
@pytest.mark.parametrize("Skv", [700, 4300])
def test_merge_types(mx, kv_type, mask, Skv):  # noqa: F811
    c = _rand_case(960 + Skv + kv_type, B=2, Sq=1, Nh=4, Nkv=2, Skv=Skv, mask=mask, kv_type=kv_type)
    check(mx, c, f"merge type {kv_type} Skv={Skv} {mask}")
