"""The decode entry points' direct host path (contiguous kernel-type operands)
against their general path: the packed argument block field by field, and on
the GPU bit-identical results over the forms it takes and no call taken that
the general path reads differently."""

import ctypes
import os
import shutil
import subprocess
import sys

import pytest
import torch

from deltanet_tpu_amd import (_lib, delta_rule_decode_step, gdn2, gdn2_decode_step, gdn2_decode_steps,
                              gla_decode_step)


def test_packed_block_has_the_struct_layout():
    a = _lib.DecodeArgs()
    vals = []
    for i, (name, t) in enumerate(a._fields_):
        v = float(i + 1) if t is ctypes.c_float else (i + 1) * 1000003
        setattr(a, name, v)
        vals.append(v)
    assert _lib.DECODE_PACK(*vals) == bytes(a)


def test_packed_entries_are_the_loaded_library(tmp_path, monkeypatch):
    # a library rebuilt under a running process stays the one that was loaded
    # (its error text and its caches are its own)
    lib = _lib.load_library()
    other = tmp_path / _lib.LIB_NAME
    shutil.copy(_lib.LIB_PATH, other)
    monkeypatch.setattr(_lib, "LIB_PATH", str(other))
    monkeypatch.setattr(_lib, "_packed", None)
    address = lambda f: ctypes.cast(f, ctypes.c_void_p).value
    one, many = _lib.packed_decode()
    assert address(one) == address(lib.dn_decode_step) and address(many) == address(lib.dn_decode_steps)


def test_variants_with_constant_gates_go_to_the_general_path(monkeypatch):
    # gla and delta pass gates of one head, which the direct path never takes
    tried = []
    monkeypatch.setattr(gdn2, "_decode_direct", lambda *a: tried.append(a))
    z = torch.zeros(1, 2, 128)
    for step, args in ((gla_decode_step, (z, z, z, z)), (delta_rule_decode_step, (z, z, z, torch.zeros(1, 2)))):
        with pytest.raises(RuntimeError, match="runs only on a ROCm GPU"):
            step(*args, torch.zeros(1, 2, 128, 128))
    assert not tried


def test_imports_without_gpu_support():
    code = """
import torch
for name in [n for n in dir(torch._C) if n.startswith("_cuda_")]:
    delattr(torch._C, name)
import deltanet_tpu_amd
try:
    deltanet_tpu_amd.gdn2_decode_step(*[torch.zeros(1, 2, 128)] * 6, torch.zeros(1, 2, 128, 128))
except RuntimeError as e:
    assert "runs only on a ROCm GPU" in str(e), e
else:
    raise SystemExit("no error")
"""
    r = subprocess.run([sys.executable, "-c", code], env={**os.environ, "PYTHONPATH": os.path.dirname(os.path.dirname(_lib.__file__))},
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr


def operands(B, L, Hk, Hv, rank, gates, qdt, sdt, dev="cuda:0"):
    gen = torch.Generator(device=dev)
    gen.manual_seed(B + 10 * L + Hv)
    rn = lambda *s: torch.randn(*s, device=dev, generator=gen)
    seq = (L,) if rank == 4 else ()
    q, k = rn(B, *seq, Hk, 128).to(qdt), rn(B, *seq, Hk, 128).to(qdt)
    v = rn(B, *seq, Hv, 128).to(qdt)
    out = []
    for i, (form, H) in enumerate(zip(gates, (Hk, Hk, Hv))):
        shape = {"channel": (B, *seq, H, 128), "one": (B, *seq, H, 1), "scalar": (B, *seq, H), "flat": (B, H),
                 "value": (B, *seq, Hv), "flat channel": (B, H, 128), "broadcast": (B, *seq, 1)}[form]
        x = rn(*shape)
        out.append(-torch.exp(x - 1) if i == 0 else torch.sigmoid(x))
    return q, k, v, *out, (0.1 * rn(B, Hv, 128, 128)).to(sdt)


def tried(monkeypatch, fn, args, kw):
    """The call's results, and whether the direct path took it."""
    direct, seen = gdn2._decode_direct, []

    def record(*a):
        seen.append(direct(*a))
        return seen[-1]

    with monkeypatch.context() as m:
        m.setattr(gdn2, "_decode_direct", record)
        got = fn(*args, **kw)
    assert len(seen) == 1
    return got, seen[0] is not None


FORMS = [("channel",) * 3, ("scalar",) * 3, ("one", "flat", "value"), ("flat channel", "value", "channel"),
         ("broadcast", "channel", "broadcast")]


@pytest.mark.gpu
@pytest.mark.parametrize("gates", FORMS)
@pytest.mark.parametrize("rank", [3, 4])
@pytest.mark.parametrize("Hk,Hv", [(2, 4), (4, 4), (1, 2), (128, 128)])
def test_step_direct_equals_general(gates, rank, Hk, Hv, monkeypatch):
    # (with one head a (B, 1, 128) gate beside rank-4 q reads as 128 heads and is refused)
    if rank == 3 or Hk == 1:
        gates = tuple("channel" if f == "flat channel" else f for f in gates)
    for qdt, sdt, out_dt in ((torch.bfloat16, torch.bfloat16, "bf"), (torch.float32, torch.float32, None),
                             (torch.float16, torch.bfloat16, None)):
        B = 3
        args = operands(B, 1, Hk, Hv, rank, gates, qdt, sdt)
        reset = torch.tensor([True, False, True], device="cuda:0")
        kw = dict(reset=reset, qk_l2norm=True, state_dtype=torch.bfloat16 if out_dt else None)
        got, taken = tried(monkeypatch, gdn2_decode_step, args, kw)
        assert taken == (Hk > 1 and "broadcast" not in gates)   # gates of one head are left
        with monkeypatch.context() as m:
            m.setattr(gdn2, "_decode_direct", lambda *a: None)
            want = gdn2_decode_step(*args, **kw)
        for x, y in zip(got, want):
            assert x.shape == y.shape and x.dtype == y.dtype and x.stride() == y.stride()
            assert torch.equal(x, y)


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 2, 5, 6, 17])
@pytest.mark.parametrize("gates", [("channel",) * 3, ("scalar",) * 3, ("one", "scalar", "value")])
def test_steps_direct_equals_general(T, gates, monkeypatch):
    for qdt, sdt in ((torch.bfloat16, torch.bfloat16), (torch.float32, torch.float32)):
        args = operands(2, T, 2, 4, 4, gates, qdt, sdt)
        for reset in (None, torch.rand(2, T, device="cuda:0") < 0.3, torch.tensor([True, False], device="cuda:0")):
            kw = dict(reset=reset, scale=0.1, state_dtype=sdt)
            got, taken = tried(monkeypatch, gdn2_decode_steps, args, kw)
            assert taken == (reset is None or reset.dim() == 2)   # a reset per row is left
            with monkeypatch.context() as m:
                m.setattr(gdn2, "_decode_direct", lambda *a: None)
                want = gdn2_decode_steps(*args, **kw)
            for x, y in zip(got, want):
                assert x.shape == y.shape and x.dtype == y.dtype and torch.equal(x, y)


@pytest.mark.gpu
def test_what_the_direct_path_leaves(monkeypatch):
    base = operands(2, 1, 2, 4, 4, ("channel",) * 3, torch.bfloat16, torch.float32)
    direct = lambda a, **kw: gdn2._decode_direct(*a, kw.get("reset"), kw.get("scale"), True, kw.get("state_dtype"),
                                                 kw.get("out_state"), False)
    assert direct(base) is not None
    sub = lambda i, x: base[:i] + (x,) + base[i + 1:]
    q, k, v, g, b, w, st = base
    left = [sub(0, q.double()), sub(1, k.float()), sub(2, v.transpose(-1, -2).contiguous().transpose(-1, -2)),
            sub(3, g[:, :, :1]), sub(4, b.expand(2, 1, 2, 128)[:, :, :, ::2]), sub(5, w.cpu()), sub(6, st[:1]),
            sub(6, st.half()), sub(2, v[:, :, :3]), sub(0, q[..., :64])]
    for a in left:
        assert direct(a) is None
    assert direct(base, scale=torch.tensor(0.1)) is None
    assert direct(base, reset=torch.tensor([True])) is None and direct(base, reset=True) is None
    assert direct(base, state_dtype="bf16") is None
    assert direct(base, out_state=torch.empty_like(st, dtype=torch.bfloat16)) is None


@pytest.mark.gpu
@pytest.mark.parametrize("tau", [None, "large", [1000.0]])
def test_a_tau_that_is_no_number_is_refused(tau):
    for T, fn in ((1, gdn2_decode_step), (3, gdn2_decode_steps)):
        args = operands(2, T, 2, 4, 4, ("channel",) * 3, torch.bfloat16, torch.float32)
        with pytest.raises((TypeError, ValueError)):
            fn(*args, stability_tau=tau)
