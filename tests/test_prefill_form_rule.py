"""Which form a prefill call takes (64-token scan or 128-token affine form), on
both sides of the rule's lines.  The two ask for different workspace per head
and 128 tokens: 150-245 KB (scan) and 450 KB or more (long form)."""

import ctypes

import pytest

from deltanet_tpu_amd import _lib


def takes_long(B, L, Hk, Hv, kind):
    a = _lib.PrefillArgs()
    a.abi_version = _lib.DN_ABI_VERSION
    a.B, a.L, a.Hk, a.Hv, a.K, a.V, a.nt = B, L, Hk, Hv, 128, 128, L
    for n in ("q", "k", "v", "g", "b", "w", "out"):
        setattr(a, n, 256)   # (only looked at for being there)
    a.qk_dtype = a.v_dtype = _lib.DN_BF16 if kind != "fp32" else _lib.DN_F32
    a.precision = int(kind == "fp32")
    for n, heads in (("g", Hk), ("b", Hk), ("w", Hv)):
        setattr(a, n + "_dtype", _lib.DN_F32)
        setattr(a, n + "_heads", heads)
        setattr(a, n + "_chans", 1 if kind == "scalar" else 128)
    size = _lib.load_library().dn_prefill_workspace_size(ctypes.byref(a))
    assert size > 0
    return (size - B * Hv * 128 * 128 * 4) / (B * Hk * ((L + 127) // 128)) > 330e3


# (kind, batch, key heads, value heads, lengths of the scan, lengths of the long form)
@pytest.mark.parametrize("kind,B,Hk,Hv,scan,lng", [
    ("channel", 1, 1, 2, [3583], [3584, 65536]),
    ("channel", 1, 4, 4, [2815], [2816, 8192, 16384]),
    ("channel", 1, 5, 10, [3583, 6657, 8191], [4096, 6144, 8192]),   # one round of 256 units: up to 6528 tokens
    ("channel", 5, 1, 2, [3583, 6657, 8191], [4096, 6144, 8192]),
    ("channel", 1, 6, 6, [2815, 5505, 6144], [3072, 5120, 8192]),
    ("channel", 1, 10, 10, [2815, 3329, 12287], [3072, 12288]),
    ("channel", 1, 12, 24, [2048, 4096, 12287], [12288, 16384]),
    ("channel", 1, 17, 17, [2048, 16384, 32768], []),
    ("channel", 1, 4, 16, [5120, 12288], [16384]),
    ("channel", 1, 3, 24, [8192], [16384]),
    ("fp32", 1, 1, 1, [3071], [3072]),
    ("fp32", 1, 8, 8, [3071, 4097], [3072, 4096, 8192]),
    ("fp32", 1, 11, 11, [4096, 8192, 16384], []),
    ("scalar", 1, 2, 2, [5119], [5120, 32768]),
    ("scalar", 1, 4, 4, [5119, 8193, 16383, 16385], [5120, 8192, 16384, 49152]),
    ("scalar", 1, 5, 5, [5119, 6657, 16384, 32768], [6144, 39297]),
    ("scalar", 1, 8, 8, [4096, 16384, 32768], []),
])
def test_lines(kind, B, Hk, Hv, scan, lng):
    assert [takes_long(B, L, Hk, Hv, kind) for L in scan] == [False] * len(scan)
    assert [takes_long(B, L, Hk, Hv, kind) for L in lng] == [True] * len(lng)
