"""Large W4A16 calls: weights unpacked to bf16 in the workspace, against the int4 kernels.

Both routes multiply the same bf16 weights ((q - z) * s exact in fp32, rounded once)
and sum in fp32, so a call with the full workspace and one without room for the
weights agree within one bf16 ulp of the output (up to 2^-7 of the value, at the foot
of a binade; 1e-3 more for values near zero, where the sums' order shows).
V of one-hot activations is a weight itself: exact, every word position and group
edge of the unpacking.  Sizes: a partial last word tile (hidden 4160: 520 words of 64
per tile), groups of 64, 192 and 128 that do not start with the tiles, both scale
types, all three projections' column offsets, head_dim 64, and with the input norm.
"""
from __future__ import annotations

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(T, hidden, Hq, Hkv, group, scale, D, norm, seed, device, onehot=False):
    from mqk import _native
    lib = _native.library()
    g = torch.Generator(device=device).manual_seed(seed)
    heads = (Hq, Hkv, Hkv)
    w = [(torch.randint(-2**31, 2**31 - 1, (hidden // 8, h * D), generator=g, device=device).int(),
          (0.005 + 0.015 * torch.rand(hidden // group, h * D, generator=g, device=device)).to(scale),
          torch.randint(-2**31, 2**31 - 1, (hidden // group, h * D // 8), generator=g, device=device).int())
         for h in heads]
    x = torch.randn(T, hidden, generator=g, device=device).bfloat16()
    if onehot:
        x = torch.zeros(T, hidden, device=device).bfloat16()
        x[torch.arange(T, device=device), torch.arange(T, device=device) % hidden] = 1.0
    gam = (1 + 0.3 * torch.randn(hidden, generator=g, device=device)).bfloat16()
    gq, gk = ((1 + 0.1 * torch.randn(D, generator=g, device=device)).bfloat16() for _ in range(2))
    cos, sin = (torch.randn(T, D, generator=g, device=device).bfloat16() for _ in range(2))
    ext = _native.FusedExt(in_gamma=gam.data_ptr(), in_eps=1e-6) if norm else _native.FusedExt()
    full = _native.fused_workspace_bytes(T, Hq, Hkv, hidden, D, ext, int4=True)
    small = _native.fused_workspace_bytes(T, Hq, Hkv, hidden, D, ext)

    def run(nbytes):
        ws = torch.zeros(max(nbytes, 256), dtype=torch.uint8, device=device)
        out = [torch.zeros(T, h, D, dtype=torch.bfloat16, device=device) for h in heads]
        st = lib.mqk_fused_qkv_rope_ex_w4a16(
            x.data_ptr(), *(t.data_ptr() for trio in w for t in trio), group,
            _native.MQK_SCALE_FP16 if scale == torch.float16 else _native.MQK_SCALE_BF16, gq.data_ptr(), gk.data_ptr(),
            cos.data_ptr(), sin.data_ptr(), None, T, T, hidden, Hq, Hkv, D, T, 1e-6, *(o.data_ptr() for o in out),
            ctypes.byref(ext), ws.data_ptr(), nbytes, int(torch.cuda.current_stream().cuda_stream))
        _native.check(st, "ex_w4a16")
        torch.cuda.synchronize()
        return out
    return run, full, small, w


@pytest.mark.parametrize("T,hidden,Hq,Hkv,group,scale,D,norm", [
    (1200, 4160, 32, 8, 64, torch.float16, 128, False), (1537, 4608, 18, 15, 192, torch.bfloat16, 128, False),
    (1300, 4096, 64, 16, 128, torch.float16, 64, False), (1025, 5120, 40, 8, 128, torch.bfloat16, 128, True),
    (3000, 2048, 32, 4, 128, torch.float16, 128, True)])
def test_unpacked_route_matches_the_int4_kernels(T, hidden, Hq, Hkv, group, scale, D, norm, device):
    run, full, small, _ = _case(T, hidden, Hq, Hkv, group, scale, D, norm, T + hidden, device)
    N = (Hq + 2 * Hkv) * D
    assert full >= small + N * hidden * 2, "the call is large enough to unpack its weights"
    a, b = run(full), run(small)
    for name, o, r in zip("qkv", a, b):
        o, r = o.float(), r.float()
        assert torch.isfinite(o).all()
        bad = (o - r).abs() > 2.0 ** -7 * r.abs() + 1e-3
        assert not bool(bad.any()), f"{name}: {int(bad.sum())} differ, max {float((o - r).abs().max())}"


def test_unpacked_weights_are_exact(device):
    """One-hot activations read every weight of V out: bit for bit the dequantised
    weight rounded to bf16."""
    T, hidden, Hq, Hkv, group, D = 4160, 4160, 2, 6, 64, 128
    run, full, small, w = _case(T, hidden, Hq, Hkv, group, torch.float16, D, False, 9, device, onehot=True)
    assert full > small
    v = run(full)[2].reshape(T, Hkv * D)
    qw, sc, qz = w[2]
    shift = torch.arange(0, 32, 4, device=device, dtype=torch.int32)
    q = ((qw[:, None, :] >> shift[None, :, None]) & 15).reshape(hidden, Hkv * D).double()
    z = ((qz[:, :, None] >> shift) & 15).reshape(hidden // group, Hkv * D).double().repeat_interleave(group, 0)
    want = ((q - z) * sc.double().repeat_interleave(group, 0)).bfloat16()
    assert torch.equal(v, want)


def test_small_calls_keep_the_int4_kernels(device):
    """The size query makes no room for unpacked weights below the planner's line (nor at
    hidden 1024).  The line is not the crossover: unpacking would pay for some of the
    calls just below it."""
    from mqk import _native
    for T, Hq, Hkv, hidden in ((768, 40, 8, 5120), (64, 32, 8, 4096), (8214, 16, 8, 1024)):
        assert _native.fused_workspace_bytes(T, Hq, Hkv, hidden, 128, int4=True) == \
            _native.fused_workspace_bytes(T, Hq, Hkv, hidden, 128)
