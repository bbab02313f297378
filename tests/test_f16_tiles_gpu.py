"""The fp16 front on the pipelined tile and decode kernels, against the 64-bit composition.

Products of fp16 values are exact in fp32 and the sums are fp32, so an output is the
64-bit value rounded once to fp16 (half an ulp, 2^-11 of the value) up to the fp32
summation error: hidden * 2^-24 of the sum of the products' magnitudes bounds it, and
sqrt(hidden) * 2^-24 is typical; relative to a projection of N(0, 1) inputs by
N(0, 0.02) weights, whose terms' magnitudes add up to about 0.64 * sqrt(hidden) of its
rms, 1e-3 of an output's rms covers it after the norm and the rotation (a sum of two
products).  Sizes: one token, the row edges of every tile (64, 128, 192, 256 rows),
head counts that each tile width divides, and head_dim 64.
"""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(B, S, hidden, Hq, Hkv, D, rows, seed, device):
    g = torch.Generator(device=device).manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g, device=device)
    x = rnd(B, S, hidden).half()
    ws = [(0.02 * rnd(h * D, hidden)).half() for h in (Hq, Hkv, Hkv)]
    gq, gk = ((1 + 0.1 * rnd(D)).half() for _ in range(2))
    ang = torch.arange(rows, device=device)[:, None] * 1e6 ** (-torch.arange(0, D, 2, device=device) / D)[None]
    ang = torch.cat([ang, ang], -1)
    return x, *ws, gq, gk, ang.cos().half(), ang.sin().half()


def _exact(x, wq, wk, wv, gq, gk, cos, sin, pos, D):
    B, S, hidden = x.shape
    x2 = x.reshape(B * S, hidden).double()
    at = torch.arange(B * S, device=x.device) % S if pos is None else pos.long()
    c, s = cos.double()[at][:, None], sin.double()[at][:, None]

    def nr(w, g):
        p = (x2 @ w.double().T).reshape(B * S, -1, D)
        n = p * torch.rsqrt(p.square().mean(-1, keepdim=True) + 1e-6) * g.double()
        return n * c + torch.cat([-n[..., D // 2:], n[..., :D // 2]], -1) * s
    return nr(wq, gq), nr(wk, gk), (x2 @ wv.double().T).reshape(B * S, -1, D)


def _check(out, ref, label):
    for name, o, r in zip("qkv", out, ref):
        assert o.dtype == torch.float16
        o = o.double().reshape(r.shape)
        rms = r.square().mean().sqrt()
        bad = (o - r).abs() > 2.0 ** -11 * r.abs() + 1e-3 * rms
        assert not bool(bad.any()), f"{label} {name}: {int(bad.sum())} beyond the bound, max {float((o - r).abs().max())}"


@pytest.mark.parametrize("B,S,hidden,Hq,Hkv,D,positions", [
    (1, 1, 64, 1, 1, 128, False), (1, 1, 4096, 32, 8, 128, True), (16, 1, 1024, 16, 8, 128, True),
    (17, 1, 1024, 16, 8, 128, True), (33, 1, 5120, 40, 8, 128, True), (64, 1, 4096, 32, 8, 128, True),
    (1, 65, 1024, 16, 8, 128, False),
    (1, 129, 2048, 32, 4, 128, False), (3, 171, 1024, 7, 2, 128, False), (1, 777, 4096, 32, 8, 128, False),
    (1, 1025, 4096, 32, 8, 128, False), (1, 1537, 4096, 32, 8, 128, False), (1, 2049, 2048, 32, 4, 128, False),
    (5, 1, 1024, 16, 8, 64, True), (2, 300, 2048, 32, 8, 64, False), (1, 1300, 1024, 12, 4, 64, False),
    (1, 70, 2080, 2, 1, 128, False)])
def test_f16_matches_the_composition(B, S, hidden, Hq, Hkv, D, positions, device):
    import mqk
    rows = 4096 if positions else S
    args = _inputs(B, S, hidden, Hq, Hkv, D, rows, 900 + B * S + hidden, device)
    pos = None
    if positions:
        pos = torch.randint(0, rows, (B * S,), generator=torch.Generator().manual_seed(B), dtype=torch.int32).to(device)
    out = mqk.fused_qkv_rope(*args, pos)
    torch.cuda.synchronize()
    _check(out, _exact(*args, pos, D), f"f16 B={B} S={S} hidden={hidden} {Hq}/{Hkv} D={D}")


@pytest.mark.parametrize("variant", [16, 18, 20, 21, 23, 25, 26, 28])
def test_f16_tile_variants(variant, device):
    """Every tile variant with an fp16 form, with a partial last row tile (T = 600) and
    30 heads (whole tiles of 1, 2, 3 and 5 heads)."""
    import mqk
    args = _inputs(2, 300, 1024, 22, 4, 128, 300, 1300 + variant, device)
    mqk.set_option("prefill_tile", variant)
    try:
        out = mqk.fused_qkv_rope(*args)
        torch.cuda.synchronize()
    finally:
        mqk.set_option("prefill_tile", 0)
    _check(out, _exact(*args, None, 128), f"f16 variant {variant}")


def test_f16_without_a_workspace(device):
    """The entry point without a workspace (no pair tiles, no split-K): the same bound."""
    from mqk import _native
    lib = _native.library()
    for T, hidden, Hq, Hkv in ((40, 4096, 32, 8), (1024, 4096, 32, 8)):
        args = _inputs(1, T, hidden, Hq, Hkv, 128, T, 1400 + T, device)
        out = [torch.zeros(T, h, 128, dtype=torch.float16, device=device) for h in (Hq, Hkv, Hkv)]
        st = lib.mqk_fused_qkv_rope_f16(*(a.data_ptr() for a in args), None, T, T, hidden, Hq, Hkv, 128, T, 1e-6,
                                        *(o.data_ptr() for o in out), int(torch.cuda.current_stream().cuda_stream))
        _native.check(st, "f16")
        torch.cuda.synchronize()
        _check(out, _exact(*args, None, 128), f"f16 no workspace T={T}")


def test_f16_large_values_saturate_like_a_cast(device):
    """V outputs past fp16's range round to infinity as a cast does, and stay out of
    the other tokens' rows."""
    import mqk
    args = list(_inputs(1, 70, 1024, 16, 8, 128, 70, 1500, device))
    args[0][0, 3] = 6e4
    args[3][:] = 1.0
    out = mqk.fused_qkv_rope(*args)
    torch.cuda.synchronize()
    ref = _exact(*args, None, 128)[2].half()
    assert bool(torch.isinf(out[2][0, 3]).all()) and bool(torch.isinf(ref[3]).all())
    assert bool(torch.isfinite(out[2][0, [0, 2, 4, 69]]).all())


@pytest.mark.parametrize("tile", [1, 16, 18, 24, 25, 28, 31])
def test_a_requested_variant_never_refuses_fp16(tile, device):
    """prefill_tile names a bf16 or int4 tile: an fp16 call whose head count, workspace or
    element type that variant does not take runs the automatic choice (the same bits: the
    tiles sum in one order)."""
    import mqk
    from mqk import _native
    T, hidden, Hq, Hkv = 200, 256, 3, 1  # (5 blocks: whole tiles for 20, 21, 25 and 27 only)
    g = torch.Generator(device=device).manual_seed(tile)
    r = lambda *s: torch.randn(*s, generator=g, device=device).half()
    args = (r(1, T, hidden), *(0.05 * r(h * 128, hidden) for h in (Hq, Hkv, Hkv)), 1 + 0.1 * r(128), 1 + 0.1 * r(128),
            r(T, 128), r(T, 128))
    lib = _native.library()
    out = [torch.zeros(T, h, 128, dtype=torch.float16, device=device) for h in (Hq, Hkv, Hkv)]
    want = mqk.fused_qkv_rope(*args)
    old = mqk.get_option("prefill_tile")
    mqk.set_option("prefill_tile", tile)
    try:
        got = mqk.fused_qkv_rope(*args)
        st = lib.mqk_fused_qkv_rope_f16(*(t.data_ptr() for t in args), None, T, T, hidden, Hq, Hkv, 128, T, 1e-6,
                                        *(o.data_ptr() for o in out), int(torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
    finally:
        mqk.set_option("prefill_tile", old)
    _native.check(st, "f16")
    for a, b, c in zip(got, want, out):
        assert torch.equal(a, b) and torch.equal(c.reshape(b.shape), b)
