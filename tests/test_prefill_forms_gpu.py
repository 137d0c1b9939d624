"""The prefill's three forms (64-token scan, its scalar-gate variant, the
128-token affine form for few heads and many chunks) against the oracle at the
edges of their tiles, chunks and dispatch ranges."""

import numpy as np
import pytest
import torch

from deltanet_tpu_amd import chunk_gdn2
from oracle import gdn_oracle as O
from tests.gpu_common import check, oracle_prefill, round_in, to_dev
from tests._util import sig

pytestmark = pytest.mark.gpu


def run(seed, B, L, Hk, Hv, *, scalar, precision, v_dt="fp32", docs=True, init=True, fuse=False):
    rng = np.random.default_rng(seed)
    rn = rng.standard_normal
    dt = "fp32" if precision == "fp32" else "bf16"
    q, k = (round_in(rn((B, L, Hk, 128)), dt) for _ in range(2))
    v = round_in(rn((B, L, Hv, 128)), v_dt)
    if scalar:
        g = (-np.exp(rn((B, L, Hv)) - 1)).astype(np.float32)
        b = sig(rn((B, L, Hv))).astype(np.float32)
        w = sig(rn((B, L, Hv))).astype(np.float32)
    else:
        g = (rn((B, L, Hk, 128)) if fuse else -np.exp(0.39 * rn((B, L, Hk, 128)) - 1)).astype(np.float32)
        b = (rn((B, L, Hk, 128)) if fuse else sig(0.39 * rn((B, L, Hk, 128)))).astype(np.float32)
        w = (rn((B, L, Hv, 128)) if fuse else sig(0.39 * rn((B, L, Hv, 128)))).astype(np.float32)
    seg = np.sort(rng.integers(0, max(2, L // 50), (B, L)), axis=1).astype(np.int32) if docs else None
    s0 = 0.1 * rn((B, Hv, 128, 128)) if init else None
    tq = torch.float32 if dt == "fp32" else torch.bfloat16
    out, st = chunk_gdn2(to_dev(q, tq), to_dev(k, tq), to_dev(v, torch.float32 if v_dt == "fp32" else torch.bfloat16),
                         to_dev(g), to_dev(b), to_dev(w), segment_ids=to_dev(seg, torch.int32), initial_state=to_dev(s0),
                         output_final_state=True, qk_l2norm=True, is_inference=True, precision=precision,
                         fuse_prologue=fuse)
    kw = dict(segment_ids=seg, qk_l2norm=True, qk_dtype="fp32" if fuse else dt)
    if init or fuse:
        ro, rs = O.chunk_gdn2(q, k, v, g, b, w, initial_state=s0, output_final_state=True, fuse_prologue=fuse, **kw)
    else:
        ro, rs = oracle_prefill(q, k, v, g, b, w, use_c=True, **kw)
    check(out, ro, st, rs, precision, v_dt, f"L={L} scalar={scalar} {precision} {v_dt}")


# around the 16-token blocks and 64-token chunks of the scan
@pytest.mark.parametrize("L", [1, 15, 17, 63, 64, 65, 113, 128, 129, 191, 193])
@pytest.mark.parametrize("scalar,precision", [(False, "bf16"), (True, "bf16"), (False, "fp32")])
def test_scan_edges(L, scalar, precision):
    run(L, 2, L, 1, 2, scalar=scalar, precision=precision, v_dt="bf16" if precision == "bf16" and L % 2 else "fp32")


# one, two and four column tiles per workgroup (256, 512 and 520 tiles), scalar
# and channel-wise gates, 16-bit and 32-bit values, the fused prologue
@pytest.mark.parametrize("B,Hk,Hv", [(1, 16, 32), (2, 16, 32), (5, 13, 13)])
@pytest.mark.parametrize("scalar,v_dt,fuse", [(False, "bf16", False), (False, "fp32", True), (True, "bf16", False),
                                              (True, "fp32", False)])
def test_column_tiles(B, Hk, Hv, scalar, v_dt, fuse):
    run(7 * B + Hv, B, 77, Hk, Hv, scalar=scalar, precision="bf16", v_dt=v_dt, fuse=fuse)


# either side of the lengths from which few heads take the affine form (3584
# tokens here, 4096 in fp32, 5120 with scalar gates), and its chunks' edges
@pytest.mark.parametrize("L,scalar,precision", [(3071, False, "bf16"), (3072, False, "bf16"), (3200, False, "fp32"),
                                                (3073, False, "fp32"), (3583, True, "bf16"), (3584, True, "bf16"),
                                                (8191, True, "bf16"), (8193, True, "bf16"), (3583, False, "bf16"),
                                                (3584, False, "bf16"), (3585, False, "bf16"), (4095, False, "fp32"),
                                                (4096, False, "fp32"), (4097, False, "fp32"), (5119, True, "bf16"),
                                                (5120, True, "bf16")])
def test_long_form_edges(L, scalar, precision):
    run(L, 1, L, 1, 2, scalar=scalar, precision=precision, init=False)
