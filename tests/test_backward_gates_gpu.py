"""Backward with gates of one value per (token, head): those gradients against
the channel-wise path's on the same gates spread over 128 channels."""

import itertools

import pytest
import torch

from deltanet_tpu_amd import chunk_gdn2

pytestmark = pytest.mark.gpu

# Both paths take the same fp32 inputs through the same products and differ in
# the roundings of the decay factors and of the channel sums: at most 512 = 4 x
# 128 terms of 2^-24 each, and 4 operands of 2^-17 where products are split
# into bf16 pairs.  Both bounds are 3.05e-5 of a gradient's norm.
RTOL = 2.0 ** -15


def grads(L, Hk, Hv, heads, chans, spread, *, precision, v_dt, decay, docs, fuse=False, recompute=False):
    gen = torch.Generator(device="cuda").manual_seed(100 * L + 10 * Hv + sum(chans))
    rn = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    B = 2
    q, k = (torch.nn.functional.normalize(rn(B, L, Hk, 128), dim=-1) for _ in range(2))
    v = rn(B, L, Hv, 128).to(v_dt)
    raw = [rn(B, L, h, c) for h, c in zip(heads, chans)]
    if not fuse:
        raw = [-decay * raw[0].exp(), raw[1].sigmoid(), raw[2].sigmoid()]
    seg = (torch.arange(L, device="cuda") // max(1, L // docs)).to(torch.int32) if docs else None
    init = 0.1 * rn(B, Hv, 128, 128)
    d_out, d_fin = rn(B, L, Hv, 128), rn(B, Hv, 128, 128)
    leaves = [q, k, v, *raw, init]
    for t in leaves:
        t.requires_grad_(True)
    g, b, w = (t.expand(*t.shape[:3], 128) if spread else t for t in raw)
    out, fin = chunk_gdn2(q, k, v, g, b, w, segment_ids=seg, initial_state=init, output_final_state=True,
                          precision=precision, qk_l2norm=fuse, fuse_prologue=fuse,
                          recompute_states=recompute)
    return torch.autograd.grad([out, fin], leaves, [d_out.to(out.dtype), d_fin])


def compare(*a, **kw):
    one, full = grads(*a, False, **kw), grads(*a, True, **kw)
    for name, x, y in zip("q k v g b w init".split(), one, full):
        x, y = x.double(), y.double()
        err = ((x - y).norm() / y.norm()).item()
        # dv is stored in v's type: one more rounding on each side
        tol = RTOL + (2.0 ** -8 if name == "v" and kw["v_dt"] == torch.bfloat16 else 0)
        assert err <= tol, (name, err)


# chunk edges; weak decay (in-block factors) and decay far beyond 2^64 in a
# 16-token block (factors per element)
@pytest.mark.parametrize("L", [1, 17, 64, 65, 200])
@pytest.mark.parametrize("decay", [0.05, 20.0])
@pytest.mark.parametrize("precision,v_dt", [("bf16", torch.bfloat16), ("fp32", torch.float32)])
def test_scalar_gates(L, decay, precision, v_dt):
    compare(L, 2, 4, (4, 4, 4), (1, 1, 1), precision=precision, v_dt=v_dt, decay=decay, docs=3)


# every mix of one-channel and channel-wise gates, gates at the key heads, at
# the value heads and shared by all heads, the fused prologue, recomputation
@pytest.mark.parametrize("chans", [c for c in itertools.product((1, 128), repeat=3) if c != (128, 128, 128)])
@pytest.mark.parametrize("heads,fuse,recompute", [((2, 2, 4), False, False), ((4, 4, 4), True, True), ((1, 1, 1), False, False),
                                                  ((2, 4, 2), False, True)])
def test_mixed_gates(chans, heads, fuse, recompute):
    compare(130, 2, 4, heads, chans, precision="fp32", v_dt=torch.float32, decay=0.3, docs=2, fuse=fuse, recompute=recompute)


# the kernels of each mix with split-bf16 products (one decay or one per channel;
# b and w of one channel, of 128, or mixed)
@pytest.mark.parametrize("chans", [c for c in itertools.product((1, 128), repeat=3) if c != (128, 128, 128)])
def test_mixed_gates_bf16(chans):
    compare(130, 2, 4, (2, 2, 4), chans, precision="bf16", v_dt=torch.bfloat16, decay=0.3, docs=2)
