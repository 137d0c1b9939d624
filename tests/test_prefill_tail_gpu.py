"""Tokens past the last one are not read: inputs that are the front of larger
buffers give the same results whatever the rest of those buffers holds."""

import pytest
import torch

from deltanet_tpu_amd import chunk_gdn2

pytestmark = pytest.mark.gpu


def run(B, L, Hk, Hv, scalar, v_dt, precision, behind):
    gen = torch.Generator(device="cuda").manual_seed(L)
    rn = lambda *s: torch.randn(*s, generator=gen, device="cuda")

    def front(x):
        # (as much again and a chunk of rows: any row that could be reached is in the buffer)
        n = x.numel()
        buf = torch.full((2 * n + 64 * x[0, 0].numel(),), behind, dtype=x.dtype, device="cuda")
        buf[:n] = x.reshape(-1)
        return buf[:n].view(x.shape)

    dt = torch.float32 if precision == "fp32" else torch.bfloat16
    q, k = (rn(B, L, Hk, 128).to(dt) for _ in range(2))
    v = rn(B, L, Hv, 128).to(v_dt)
    chans = () if scalar else (128,)
    g, b = -torch.exp(rn(B, L, Hk, *chans) - 1), torch.sigmoid(rn(B, L, Hk, *chans))
    w = torch.sigmoid(rn(B, L, Hv, *chans))
    out, state = chunk_gdn2(*(front(x) for x in (q, k, v, g, b, w)), output_final_state=True, qk_l2norm=True,
                            is_inference=True, precision=precision)
    assert torch.isfinite(out).all() and torch.isfinite(state).all()
    return out, state


# tails of 1, 3, 15, 17 and 63 tokens behind two chunks of 64; one, two and four
# column tiles per workgroup (scalar gates with 16-bit values at four: each wave
# a tile of its own), float32, and the long form's 128-token chunks
@pytest.mark.parametrize("tail", [1, 3, 15, 17, 63])
@pytest.mark.parametrize("B,Hk,Hv,scalar,v_dt,precision,chunks", [
    (5, 13, 13, True, torch.bfloat16, "bf16", 2),
    (5, 13, 13, True, torch.float32, "bf16", 2),
    (5, 13, 13, False, torch.bfloat16, "bf16", 2),
    (2, 16, 32, True, torch.bfloat16, "bf16", 2),
    (1, 2, 4, False, torch.bfloat16, "bf16", 2),
    (1, 2, 4, False, torch.float32, "fp32", 2),
    (1, 1, 2, False, torch.bfloat16, "bf16", 56),
    (1, 1, 2, True, torch.bfloat16, "bf16", 96),
])
def test_memory_behind_the_inputs(tail, B, Hk, Hv, scalar, v_dt, precision, chunks):
    L = 64 * chunks + tail
    a = run(B, L, Hk, Hv, scalar, v_dt, precision, 0.0)
    b = run(B, L, Hk, Hv, scalar, v_dt, precision, float("nan"))
    for x, y in zip(a, b):
        assert torch.equal(x, y)
