"""The input RMSNorm's two forms: rows normalised ahead in the workspace, and (a
workspace without that room) in the projection kernels.

Both compute bf16(gamma * bf16(x * scale)) with one scale per token and run the
same MFMA order wherever they take the same plan, so a call at the C ABI with the
full workspace and one with the smallest must agree: bit for bit where the launch
is the same kernel (test_both_forms_agree_on_one_kernel requests it), and within one
bf16 ulp where it need not be (test_both_forms_agree): two differently split fp32 sums
differ by about 1e-6 of their terms, so their bf16 roundings differ by at most one ulp,
which is up to 2^-7 of the value (at the foot of a binade); 1e-3 is added for values
near zero.  At decode sizes the smallest workspace gets the decode kernel with fewer
splits and rows ahead, wherever it has more than one.
Sizes: one token, odd hidden chunk counts (hidden 192: 24 of 64 lanes hold chunks;
hidden 2112: a partial fifth chunk; 16384: a row of two passes), the block and tile
edges, and int4 weights.
"""
from __future__ import annotations

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

D = 128


def _call(T, hidden, Hq, Hkv, int4, seed, device):
    """(run(ws_bytes) -> (q, k, v), full size, smallest size)."""
    from mqk import _native
    lib = _native.library()
    g = torch.Generator(device=device).manual_seed(seed)
    x = (3 * torch.randn(T, hidden, generator=g, device=device)).bfloat16()
    gam = (1 + 0.3 * torch.randn(hidden, generator=g, device=device)).bfloat16()
    gq, gk = ((1 + 0.1 * torch.randn(D, generator=g, device=device)).bfloat16() for _ in range(2))
    cos, sin = (torch.randn(T, D, generator=g, device=device).bfloat16() for _ in range(2))
    heads = (Hq, Hkv, Hkv)
    if int4:
        w = [(torch.randint(-2**31, 2**31 - 1, (hidden // 8, h * D), generator=g, device=device).int(),
              (0.005 + 0.015 * torch.rand(hidden // 64, h * D, generator=g, device=device)).half(),
              torch.randint(-2**31, 2**31 - 1, (hidden // 64, h * D // 8), generator=g, device=device).int())
             for h in heads]
        flat = [t.data_ptr() for trio in w for t in trio] + [64, _native.MQK_SCALE_FP16]
    else:
        w = [(0.02 * torch.randn(h * D, hidden, generator=g, device=device)).bfloat16() for h in heads]
        flat = [t.data_ptr() for t in w]
    ext = _native.FusedExt(in_gamma=gam.data_ptr(), in_eps=1e-6)
    full = int(lib.mqk_fused_qkv_rope_ex_workspace_size(T, Hq, Hkv, hidden, ctypes.byref(ext)))
    least = _native.least_workspace_bytes(T, Hq, Hkv, hidden, D, ext)
    entry = lib.mqk_fused_qkv_rope_ex_w4a16 if int4 else lib.mqk_fused_qkv_rope_ex_bf16

    def run(nbytes):
        ws = torch.zeros(nbytes, dtype=torch.uint8, device=device)
        out = [torch.zeros(T, h, D, dtype=torch.bfloat16, device=device) for h in heads]
        stream = int(torch.cuda.current_stream().cuda_stream)
        st = entry(x.data_ptr(), *flat, gq.data_ptr(), gk.data_ptr(), cos.data_ptr(), sin.data_ptr(), None, T, T,
                   hidden, Hq, Hkv, D, T, 1e-6, *(o.data_ptr() for o in out), ctypes.byref(ext), ws.data_ptr(), nbytes,
                   stream)
        _native.check(st, "ex")
        torch.cuda.synchronize()
        # the arrival counters (their statistics word aside) are zero again
        words = ws[: _native._COUNTER_BYTES].view(torch.int32)
        assert int(words[:1024].abs().sum()) == 0 and int(words[1024 + 64:].abs().sum()) == 0
        return out, (x, w, gam)
    return run, full, least


@pytest.mark.parametrize("T,hidden,Hq,Hkv,int4", [
    (1, 192, 2, 1, False), (3, 2112, 4, 2, False), (64, 1024, 16, 8, False), (65, 1024, 16, 8, False),
    (129, 16384, 2, 1, False), (333, 2048, 32, 4, False), (700, 4096, 32, 8, False),
    (1, 192, 2, 1, True), (17, 4096, 32, 8, True), (70, 1024, 16, 8, True), (257, 2048, 32, 4, True)])
def test_both_forms_agree(T, hidden, Hq, Hkv, int4, device):
    run, full, least = _call(T, hidden, Hq, Hkv, int4, 77 + T + hidden, device)
    assert full > least
    ahead, _ = run(full)
    staged, _ = run(least)
    for name, a, b in zip("qkv", ahead, staged):
        a, b = a.float(), b.float()
        assert torch.isfinite(a).all()
        assert bool(((a - b).abs() <= 2.0 ** -7 * b.abs() + 1e-3 * b.square().mean().sqrt().clamp(min=1.0)).all()), name


def test_rows_are_the_rounded_norm(device):
    """One-hot V rows copy normalised activations out: the 64-bit norm rounded twice
    to bf16, except where the fp32 scale's last bits flip the first rounding (under
    0.5 % of them): one ulp there, and the product with gamma (below 2) can make it
    two."""
    T, hidden, Hq, Hkv = 40, 1024, 2, 8
    import mqk
    g = torch.Generator(device=device).manual_seed(5)
    x = (3 * torch.randn(1, T, hidden, generator=g, device=device)).bfloat16()
    gam = (1 + 0.3 * torch.randn(hidden, generator=g, device=device)).bfloat16()
    wq = torch.randn(Hq * D, hidden, generator=g, device=device).bfloat16()
    wk = torch.randn(Hkv * D, hidden, generator=g, device=device).bfloat16()
    wv = torch.eye(hidden, device=device).bfloat16()
    one = torch.ones(D, dtype=torch.bfloat16, device=device)
    cos = torch.ones(T, D, dtype=torch.bfloat16, device=device)
    _, _, v = mqk.fused_qkv_rope_ex(x, wq, wk, wv, one, one, cos, cos, input_norm_w=gam)
    xd = x[0].double()
    y = (xd * torch.rsqrt(xd.square().mean(-1, keepdim=True) + 1e-6)).bfloat16()
    want = (gam.double() * y.double()).bfloat16()
    diff = (v.reshape(T, hidden).view(torch.int16).int() - want.view(torch.int16).int()).abs()
    assert int(diff.max()) <= 2 and float((diff > 0).float().mean()) < 5e-3


def test_capture_in_a_workspace_of_the_scales_only(device):
    """Captured with a buffer that holds the plan and the per-token scales but not
    the rows: the call is accepted and replays (it was before rows were written
    ahead), with the eager call's values."""
    import mqk
    from mqk import _native
    T, hidden, Hq, Hkv = 64, 1024, 16, 8
    g = torch.Generator(device=device).manual_seed(6)
    ws = [(0.02 * torch.randn(h * D, hidden, generator=g, device=device)).bfloat16() for h in (Hq, Hkv, Hkv)]
    one = torch.ones(D, dtype=torch.bfloat16, device=device)
    cos = torch.randn(T, D, generator=g, device=device).bfloat16()
    gam = (1 + 0.3 * torch.randn(hidden, generator=g, device=device)).bfloat16()
    x = torch.randn(1, T, hidden, generator=g, device=device).bfloat16()
    call = lambda: mqk.fused_qkv_rope_ex(x, *ws, one, one, cos, cos, input_norm_w=gam)
    want = call()
    stream = torch.cuda.Stream(device)
    ext = _native.FusedExt(in_gamma=gam.data_ptr(), in_eps=1e-6)
    least = _native.least_workspace_bytes(T, Hq, Hkv, hidden, D, ext)
    with torch.cuda.stream(stream):
        _native._workspaces[(device.index or 0, int(stream.cuda_stream))] = torch.zeros(least, dtype=torch.uint8,
                                                                                       device=device)
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            out = call()
    for _ in range(3):
        for t in out:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(out, want):
            assert bool(((a.float() - b.float()).abs() <= 2.0 ** -7 * b.float().abs() + 1e-3).all())
    _native._workspaces.pop((device.index or 0, int(stream.cuda_stream)))


@pytest.mark.parametrize("T,hidden,heads,kv,D,int4", [
    (1100, 3072, 40, 10, 64, False),  # the size query plans pair tiles, the call the split-K launch: ten times the bytes
    (777, 4096, 64, 16, 64, False), (900, 2048, 48, 24, 64, False), (130, 4096, 64, 16, 64, False), (500, 8448, 20, 5, 128, False),
    (1000, 4096, 32, 8, 128, False), (300, 2048, 32, 4, 128, False), (40, 1024, 16, 8, 64, False),
    (777, 4096, 64, 16, 64, True), (130, 1024, 16, 8, 128, True), (1300, 4096, 64, 16, 64, True)])
def test_rows_are_written_ahead_at_the_queried_size(T, hidden, heads, kv, D, int4, device):
    """A workspace of exactly the queried bytes holds the normalised rows at its end
    (before the unpacked weights of a large int4 call), whatever plan the call takes, and
    the outputs are the plain call's on those rows in what is left of it, bit for bit."""
    from mqk import _native
    lib = _native.library()
    g = torch.Generator(device=device).manual_seed(T + hidden)
    r = lambda *s: torch.randn(*s, generator=g, device=device)
    x, gam = (3 * r(T, hidden)).bfloat16(), (1 + 0.3 * r(hidden)).bfloat16()
    gq, gk = ((1 + 0.1 * r(D)).bfloat16() for _ in range(2))
    cos, sin = (r(T, D).bfloat16() for _ in range(2))
    counts = (heads, kv, kv)
    if int4:
        w = [t for h in counts for t in
             (torch.randint(-2**31, 2**31 - 1, (hidden // 8, h * D), generator=g, device=device).int(),
              (0.005 + 0.015 * torch.rand(hidden // 64, h * D, generator=g, device=device)).half(),
              torch.randint(-2**31, 2**31 - 1, (hidden // 64, h * D // 8), generator=g, device=device).int())]
        flat = [t.data_ptr() for t in w] + [64, _native.MQK_SCALE_FP16]
    else:
        w = [(0.02 * r(h * D, hidden)).bfloat16() for h in counts]
        flat = [t.data_ptr() for t in w]
    ext = _native.FusedExt(in_gamma=gam.data_ptr(), in_eps=1e-6)
    full = _native.fused_workspace_bytes(T, heads, kv, hidden, D, ext, int4=int4)
    entry = lib.mqk_fused_qkv_rope_ex_w4a16 if int4 else lib.mqk_fused_qkv_rope_ex_bf16

    def run(rows_in, e, ws, nbytes):
        out = [torch.zeros(T, h, D, dtype=torch.bfloat16, device=device) for h in counts]
        st = entry(rows_in.data_ptr(), *flat, gq.data_ptr(), gk.data_ptr(), cos.data_ptr(), sin.data_ptr(), None, T, T,
                   hidden, heads, kv, D, T, 1e-6, *(o.data_ptr() for o in out), ctypes.byref(e), ws.data_ptr(), nbytes,
                   int(torch.cuda.current_stream().cuda_stream))
        _native.check(st, "ex")
        torch.cuda.synchronize()
        return out

    ws = torch.zeros(full, dtype=torch.uint8, device=device)
    out = run(x, ext, ws, full)
    wbytes = sum(h * D for h in counts) * hidden * 2 if full > _native.fused_workspace_bytes(T, heads, kv, hidden, D, ext) else 0
    nrows = T * hidden * 2
    at = (full - wbytes & ~255) - (nrows + 255) // 256 * 256
    rows = ws[at:at + nrows].view(torch.bfloat16).reshape(T, hidden).clone()
    y = (x.double() * torch.rsqrt(x.double().square().mean(-1, keepdim=True) + 1e-6)).bfloat16()
    want = (gam.double() * y.double()).bfloat16()
    ulps = (rows.view(torch.int16).int() - want.view(torch.int16).int()).abs()
    assert int(ulps.max()) <= 2 and float((ulps > 0).float().mean()) < 5e-3  # (see test_rows_are_the_rounded_norm)
    left = at + wbytes  # (the plain call's weights again at the end of what it is given)
    plain = run(rows, _native.FusedExt(), torch.zeros(left, dtype=torch.uint8, device=device), left)
    for name, a, b in zip("qkv", out, plain):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16)), name


def test_more_rows_than_are_written_ahead(device):
    """Above 256 MiB of rows the projection kernels normalise what they stage, with the
    plain plan's pair tiles and the rows past its last whole tile on the decode kernel
    (which reads those few rows ahead).  Every row must be the row of a call that writes
    it ahead: the same bits on the tiles, one bf16 ulp on the decode rows, whose sums are
    split differently."""
    import mqk
    from conftest import launched_kernels
    T, hidden, Hq, Hkv, tail = 32768 + 22, 5120, 9, 3, 22
    g = torch.Generator(device=device).manual_seed(3)
    w = [(0.02 * torch.randn(h * D, hidden, generator=g, device=device)).bfloat16() for h in (Hq, Hkv, Hkv)]
    one = torch.ones(D, dtype=torch.bfloat16, device=device)
    cos, sin = (torch.randn(4096, D, generator=g, device=device).bfloat16() for _ in range(2))
    gam = (1 + 0.3 * torch.randn(hidden, generator=g, device=device)).bfloat16()
    x = torch.randn(1, T, hidden, generator=g, device=device).bfloat16()
    pos = torch.randint(0, 4096, (T,), generator=g, device=device).int()
    call = lambda a, b: mqk.fused_qkv_rope_ex(x[:, a:b], *w, one, one, cos, sin, pos[a:b], input_norm_w=gam)
    assert launched_kernels(lambda: call(0, T)) == ["row_scale", "row_scale", "tile_pair", "decode"]
    out = call(0, T)
    for a in range(0, T, 16384):
        b = min(a + 16384, T)
        for name, o, r in zip("qkv", out, call(a, b)):
            o = o[:, a:b]
            if b == T:
                o, r = o[:, -tail:].float(), r[:, -tail:].float()
                assert bool(((o - r).abs() <= 2.0 ** -7 * r.abs() + 1e-3).all()), name
            else:
                assert torch.equal(o.view(torch.int16), r.view(torch.int16)), name
    mqk.set_option("prefill_tile", 25)  # (the planned pair tiles: accepted by name too)
    try:
        tiles = call(0, T)
        torch.cuda.synchronize()
    finally:
        mqk.set_option("prefill_tile", 0)
    for name, o, r in zip("qkv", tiles, out):
        assert torch.equal(o[:, :-tail].view(torch.int16), r[:, :-tail].view(torch.int16)), name
    torch.cuda.synchronize()
    mqk.release_workspaces(retired_only=False)


@pytest.mark.parametrize("tile", [16, 24, 25])
@pytest.mark.parametrize("T", [2048, 2078])
def test_both_forms_agree_on_one_kernel(T, tile, device):
    """With one tile variant requested, the call with rows written ahead and the one with
    their scales only give the same bits (but for rows that go to the decode kernel)."""
    import mqk
    Hq, Hkv = (20, 5) if tile == 25 else (32, 8)
    mqk.set_option("prefill_tile", tile)
    mqk.set_option("tail_split", 0)
    try:
        run, full, least = _call(T, 1024, Hq, Hkv, False, 5, device)
        (ahead, _), (staged, _) = run(full), run(least)
    finally:
        mqk.set_option("prefill_tile", 0)
        mqk.set_option("tail_split", 1)
    for name, a, b in zip("qkv", ahead, staged):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16)), name


@pytest.mark.parametrize("T,hidden,Hq,Hkv,int4", [(1, 1024, 16, 8, False), (16, 4096, 32, 8, False),
                                                  (64, 4096, 32, 8, False), (24, 5120, 40, 8, False),
                                                  (8, 4096, 32, 8, True), (64, 2048, 32, 4, True)])
def test_decode_with_the_least_workspace(T, hidden, Hq, Hkv, int4, device):
    """Decode sizes in a workspace of the plain size and the scales: still the decode
    kernel, on rows written ahead beside the partials of fewer splits."""
    from conftest import launched_kernels
    run, full, least = _call(T, hidden, Hq, Hkv, int4, 11 + T, device)
    assert launched_kernels(lambda: run(least)) == ["row_scale", "decode"]
    for name, a, b in zip("qkv", run(full)[0], run(least)[0]):
        a, b = a.float(), b.float()
        assert bool(((a - b).abs() <= 2.0 ** -7 * b.abs() + 1e-3 * b.square().mean().sqrt().clamp(min=1.0)).all()), name
