"""Captured calls whose workspace only makes them faster: fp16 tensors and W4A16 calls that
unpack their weights.

Their graphs share nothing with the capture stream or with each other: the workspace is the
graph's own memory.  Each graph is replayed several times, with eager calls between, and
two graphs captured on one stream at once on two streams; every replay must give the eager
call's bits, and the stream's workspace must not be touched.
"""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

D = 128


def _f16(seed, T, device):
    import mqk
    hidden, Hq, Hkv = 1024, 16, 8
    g = torch.Generator(device=device).manual_seed(seed)
    r = lambda *s, std=1.0: (std * torch.randn(*s, generator=g, device=device)).half()
    args = (r(1, T, hidden), *(r(h * D, hidden, std=0.02) for h in (Hq, Hkv, Hkv)), 1 + r(D, std=0.1), 1 + r(D, std=0.1),
            r(T, D), r(T, D))
    return lambda: mqk.fused_qkv_rope(*args)


def _w4(seed, T, device, norm=False):
    import mqk
    hidden, Hq, Hkv = 4096, 32, 8
    g = torch.Generator(device=device).manual_seed(seed)
    w = [(torch.randint(-2**31, 2**31 - 1, (hidden // 8, h * D), generator=g, device=device).int(),
          (0.005 + 0.015 * torch.rand(hidden // 128, h * D, generator=g, device=device)).half(),
          torch.randint(-2**31, 2**31 - 1, (hidden // 128, h * D // 8), generator=g, device=device).int())
         for h in (Hq, Hkv, Hkv)]
    r = lambda *s: torch.randn(*s, generator=g, device=device).bfloat16()
    one = torch.ones(D, dtype=torch.bfloat16, device=device)
    x, cos, sin = r(1, T, hidden), r(T, D), r(T, D)
    gam = 1 + 0.1 * r(hidden) if norm else None
    return lambda: mqk.fused_qkv_rope_w4a16_ex(x, *w, one, one, cos, sin, input_norm_w=gam)


CASES = {"f16-decode": lambda s, d: _f16(s, 8, d), "f16-pair": lambda s, d: _f16(s, 3000, d),
         "unpack": lambda s, d: _w4(s, 1300, d), "unpack-norm": lambda s, d: _w4(s, 1300, d, True)}


@pytest.mark.parametrize("front", [True, False])
@pytest.mark.parametrize("make", CASES.values(), ids=CASES.keys())
def test_graphs_are_independent(make, front, device, monkeypatch):
    from mqk import _native
    if not front:
        monkeypatch.setattr(_native, "_front", None)
        monkeypatch.setattr(_native, "_front_absent", True)
    fns = [make(s, device) for s in (1, 2)]
    want = [fn() for fn in fns]
    capture, other = torch.cuda.Stream(device), torch.cuda.Stream(device)
    key = (device.index or 0, int(capture.cuda_stream))
    with torch.cuda.stream(capture):
        fns[0]()  # (the capture stream has a workspace that would do)
    torch.cuda.synchronize()
    shared = _native._workspaces.get(key)
    graphs, outs = [], []
    for fn in fns:
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[-1], stream=capture):
            outs.append(fn())
    assert _native._workspaces.get(key) is shared
    if shared is not None:
        shared.fill_(0x5A)  # a replay that used it would read these counters or change them
    torch.cuda.synchronize()
    for _ in range(3):
        for out in outs:
            for t in out:
                t.zero_()
        torch.cuda.synchronize()
        for g, stream in zip(graphs, (capture, other)):  # at once
            with torch.cuda.stream(stream):
                g.replay()
        torch.cuda.synchronize()
        for out, w in zip(outs, want):
            assert all(torch.equal(a, b) for a, b in zip(out, w))
        for fn, w in zip(fns, want):
            assert all(torch.equal(a, b) for a, b in zip(fn(), w))
    if shared is not None:
        assert bool((shared == 0x5A).all())
        shared.zero_()
    torch.cuda.synchronize()
