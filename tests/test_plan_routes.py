"""Which kernel a call takes and how its keys are split, seen through the host
API compiled over a stub HIP runtime (tests/c/api_host.cpp): no GPU."""
from __future__ import annotations

import ctypes
import os
import re
import shutil
import subprocess

import pytest

torch = pytest.importorskip("torch")
import mxfa  # noqa: E402

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
D = 128


@pytest.fixture(scope="module")
def api(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    so = str(tmp_path_factory.mktemp("api") / "api_host.so")
    subprocess.run([hipcc, "-x", "hip", "--offload-host-only", "--offload-arch=gfx950", "-std=c++17", "-O1", "-fPIC",
                    "-I", os.path.join(REPO, "include"), "-I", os.path.join(REPO, "acestep.cpp_amd", "csrc"), "-shared",
                    "-no-hip-rt", "-Wl,-Bsymbolic", os.path.join(REPO, "tests", "c", "api_host.cpp"), "-o", so], check=True)
    lib = ctypes.CDLL(so)
    lib.stub_log.restype = ctypes.c_char_p
    lib.mxfa_last_error.restype = ctypes.c_char_p
    return lib


def _call(api, Sq, Skv, B=1, Nh=32, Nkv=8, kv=1, mask=None, entry="mxfa_flash_attn_ext", stream=1):
    """Status and log of one call.  mask: None, or the entries per row (a dense
    mask of that pitch)."""
    row = 136 if kv == 8 else 2 * D
    T = mxfa.DeviceView
    q = T(0, (D, Sq, Nh, B), (4, 4 * D * Nh, 4 * D, 4 * D * Nh * Sq), 1 << 30).desc()
    k = T(kv, (D, Skv, Nkv, B), (34 if kv == 8 else 2, row, row * Skv, row * Skv * Nkv), 1 << 31).desc()
    v = T(kv, (D, Skv, Nkv, B), (34 if kv == 8 else 2, row, row * Skv, row * Skv * Nkv), 1 << 32).desc()
    o = T(0, (D, Nh, Sq, B), (4, 4 * D, 4 * D * Nh, 4 * D * Nh * Sq), 1 << 33).desc()
    m = mask and T(1, (mask, Sq, 1, B), (2, 2 * mask, 2 * mask * Sq, 2 * mask * Sq), 1 << 34).desc()
    p = mxfa.make_params(D ** -0.5)
    r = ctypes.byref
    args = [r(q), r(k), r(v), r(m) if m else None, r(p)] + ([] if entry == "mxfa_reserve" else [r(o)])
    rc = getattr(api, entry)(*args, ctypes.c_void_p(stream))
    return rc, api.stub_log().decode()


def _splits(log):
    return int(re.search(r"decode splits=(\d+)", log).group(1))


@pytest.fixture(autouse=True)
def fresh(api):
    api.stub_set(1 << 30, 0)
    yield
    api.stub_set(1 << 30, 0)
    api.mxfa_release()
    api.stub_log()


# 257 .. 511 streams of 16 rows: two splits where they are the faster, one elsewhere
@pytest.mark.parametrize("kv,mask,B,Sq,Skv,splits", [
    (1, 0, 5, 32, 4096, 2), (1, 4096, 5, 32, 4096, 2), (30, 0, 5, 32, 2048, 2),
    (1, 0, 5, 32, 1024, 1), (1, 0, 3, 60, 2048, 1), (1, 0, 7, 28, 2048, 2), (1, 0, 4, 40, 1024, 1),
    (8, 0, 5, 32, 4096, 2), (8, 0, 5, 32, 2048, 1), (8, 0, 7, 28, 4096, 1),
    (1, 4095, 5, 32, 4095, 2), (1, 2047, 5, 32, 2047, 1),
    (1, 0, 4, 32, 4096, 2), (1, 0, 8, 32, 8192, 1),      # 256 and 512 streams: the targets' own
])
def test_two_splits_between_the_targets(api, kv, mask, B, Sq, Skv, splits):
    rc, log = _call(api, Sq, Skv, B=B, kv=kv, mask=mask)
    assert rc == 0 and _splits(log) == splits, log


# the merge tests' split counts at one and four streams
@pytest.mark.parametrize("Skv,G,Sq,splits", [
    (66, 1, 1, 1), (130, 1, 1, 2), (68, 1, 1, 2), (132, 1, 1, 3), (68, 8, 2, 2), (132, 3, 6, 3), (2048, 1, 1, 32),
    (2100, 1, 1, 33), (4096, 1, 1, 64), (6000, 1, 1, 47), (4096, 8, 2, 64)])
def test_merge_split_counts(api, Skv, G, Sq, splits):
    rc, log = _call(api, Sq, Skv, Nh=G, Nkv=1, mask=Skv)
    assert rc == 0 and _splits(log) == splits, log


def test_two_splits_need_no_more_than_there_is(api):
    # 504 streams' partials are past the fixed scratch, 320 streams' are not
    assert _splits(_call(api, 36, 8192, B=7, entry="mxfa_flash_attn_ext_noalloc")[1]) == 1
    assert _splits(_call(api, 32, 4096, B=5, entry="mxfa_flash_attn_ext_noalloc")[1]) == 2
    # a stream whose workspace cannot grow under capture
    api.stub_set(1 << 30, 1)
    rc, log = _call(api, 32, 4096, B=5, stream=2)
    assert rc == 0 and _splits(log) == 1


# odd mask rows: the prefill kernels from where they are the faster, either side of each line of the rule
@pytest.mark.parametrize("B,Sq,Nh,Skv,decode", [
    (1, 64, 16, 4001, True), (1, 65, 16, 2047, True), (1, 65, 16, 2049, False),
    (1, 104, 16, 1001, True), (1, 105, 16, 1001, False), (1, 104, 16, 2049, False),
    (1, 208, 16, 255, True), (1, 209, 16, 255, False), (1, 208, 16, 257, False),
    (2, 256, 16, 127, True), (2, 257, 16, 127, False), (2, 256, 16, 129, False),
    (1, 127, 32, 127, True), (1, 333, 32, 333, False), (4, 127, 16, 127, True), (4, 128, 32, 41, False),
    (2, 125, 16, 41, True), (2, 1085, 16, 238, False), (1, 437, 16, 437, False),
])
@pytest.mark.parametrize("kv", [1, 30])
def test_odd_mask_rows_route(api, kv, B, Sq, Nh, Skv, decode):
    rc, log = _call(api, Sq, Skv, B=B, Nh=Nh, kv=kv, mask=Skv)
    assert rc == 0 and ("decode" in log) == decode and ("classify" in log) != decode, log
    # (rows of whole 4-value groups are not concerned)
    pitch = (Skv + 3) & ~3
    assert "decode" not in _call(api, Sq, Skv, B=B, Nh=Nh, kv=kv, mask=pitch)[1]


# (the first call's allocations: the workspace, then its tickets)
@pytest.mark.parametrize("call,runs", [
    (dict(Sq=128, Skv=1701, Nh=8, Nkv=2, B=2, mask=1701), {0: None, 1: "classify;prefill parts=0"}),
    (dict(Sq=128, Skv=1700, Nh=8, Nkv=2, mask=1700), {0: None, 1: "classify;prefill parts=0"}),
    (dict(Sq=128, Skv=1701, Nh=8, Nkv=2), {0: "wide", 1: "wide"}),
    (dict(Sq=300, Skv=333, mask=333), {0: "decode splits=1"}),
    (dict(Sq=32, Skv=4096, B=5), {0: "decode splits=1", 1: "decode splits=1"}),
    (dict(Sq=1, Skv=4096), {0: None, 1: None}),
])
def test_no_memory_falls_back(api, call, runs):
    for budget, run in runs.items():
        for entry in ("mxfa_reserve", "mxfa_flash_attn_ext"):
            api.mxfa_release()
            api.stub_set(budget, 0)
            rc, log = _call(api, entry=entry, stream=3, **call)
            assert (rc == 0) == (run is not None), (budget, entry, api.mxfa_last_error())
            assert entry == "mxfa_reserve" or run is None or log.startswith(run), (budget, log)


def test_captured_calls_fall_back(api):
    """No workspace yet and none to be had under capture: as without memory."""
    api.stub_set(1 << 30, 1)
    for entry in ("mxfa_reserve", "mxfa_flash_attn_ext"):
        assert _call(api, 300, 333, mask=333, entry=entry, stream=4)[0] == 0
        assert _call(api, 128, 1701, Nh=8, Nkv=2, entry=entry, stream=4)[0] == 0
        assert _call(api, 300, 332, mask=332, entry=entry, stream=4)[0] != 0   # aligned rows: refused, as ever
        assert _call(api, 1, 4096, entry=entry, stream=4)[0] != 0
