"""Calls of several launches from several threads on one stream.

The launches of a call hand normalised rows, scales or unpacked weights on in the stream's
workspace, which all threads that issue on the stream share.  A call's launches must
therefore reach the stream together, whichever code issues them.
"""
from __future__ import annotations

import threading

import pytest
import torch

pytestmark = pytest.mark.gpu

D = 128


def _rope(T, device):
    import mqk
    one = torch.ones(D, dtype=torch.bfloat16, device=device)
    return (one, one, *(t.bfloat16().to(device) for t in mqk.rope_tables(D, T)))


def _normed(i, T, device, D=D):
    """A call with the input norm: its rows (and no weight) differ from thread to thread."""
    import mqk
    hidden, Hq, Hkv = 1024, 4, 2
    g = torch.Generator(device=device).manual_seed(1)
    w = [(0.05 * torch.randn(h * D, hidden, generator=g, device=device)).bfloat16() for h in (Hq, Hkv, Hkv)]
    one = torch.ones(D, dtype=torch.bfloat16, device=device)
    tab = [t.bfloat16().to(device) for t in mqk.rope_tables(D, T)]
    gam = torch.ones(hidden, dtype=torch.bfloat16, device=device)
    x = (10.0 ** i * torch.randn(1, T, hidden, generator=g.manual_seed(2 + i), device=device)).bfloat16()
    return lambda: mqk.fused_qkv_rope_ex(x, *w, one, one, *tab, input_norm_w=gam)


def _unpacked(i, T, device):
    """A W4A16 call whose weights, another set in each thread, are unpacked in the workspace."""
    import mqk
    hidden, Hq, Hkv = 4096, 32, 8
    g = torch.Generator(device=device).manual_seed(7 + i)
    w = [(torch.randint(-2**31, 2**31 - 1, (hidden // 8, h * D), generator=g, device=device).int(),
          (0.005 + 0.015 * torch.rand(hidden // 128, h * D, generator=g, device=device)).half(),
          torch.randint(-2**31, 2**31 - 1, (hidden // 128, h * D // 8), generator=g, device=device).int())
         for h in (Hq, Hkv, Hkv)]
    x = torch.randn(1, T, hidden, generator=g, device=device).bfloat16()
    rope = _rope(T, device)
    return lambda: mqk.fused_qkv_rope_w4a16(x, *w, *rope)


@pytest.mark.parametrize("front", [False, True])
@pytest.mark.parametrize("make,calls", [
    (lambda i, device: _normed(i, 8, device), 300), (lambda i, device: _normed(i, 300, device), 300),
    (lambda i, device: _normed(i, 40, device, 72), 300), (lambda i, device: _unpacked(i, 1200, device), 40)],
    ids=["rows", "rows-tiles", "scales-any-head-size", "weights"])
def test_threads_on_one_stream(make, calls, front, device, monkeypatch):
    from mqk import _native
    if not front:
        monkeypatch.setattr(_native, "_front", None)
        monkeypatch.setattr(_native, "_front_absent", True)
    fns = [make(i, device) for i in range(2)]
    want = [fn() for fn in fns]
    torch.cuda.synchronize()
    wrong = torch.zeros(2, dtype=torch.int64, device=device)
    start = threading.Barrier(2)

    def work(i):
        with torch.cuda.device(device):
            start.wait()
            outs = [fns[i]()[2] for _ in range(calls)]
            for o in outs:
                wrong[i] += (o.view(torch.int16) != want[i][2].view(torch.int16)).any()
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert wrong.tolist() == [0, 0], "calls with another thread's rows or weights"


def test_the_front_lets_other_threads_run(device):
    """The C++ front releases the GIL around its allocations and launches: with a switch
    interval that no thread outwaits, another Python thread gets on only while a call
    waits for the driver."""
    import sys
    from mqk import _native
    import mqk
    ext = _native.front()
    hidden, Hq, Hkv, T = 256, 2, 1, 4
    w = [torch.zeros(h * D, hidden, dtype=torch.bfloat16, device=device) for h in (Hq, Hkv, Hkv)]
    x = torch.zeros(1, T, hidden, dtype=torch.bfloat16, device=device)
    gam = torch.ones(hidden, dtype=torch.bfloat16, device=device)
    int4 = [(torch.zeros(hidden // 8, h * D, dtype=torch.int32, device=device),
             torch.ones(2, h * D, dtype=torch.float16, device=device),
             torch.zeros(2, h * D // 8, dtype=torch.int32, device=device)) for h in (Hq, Hkv, Hkv)]
    rope = _rope(T, device)
    opt = (None, None, None, gam, 1e-6) + (None,) * 5 + (True,)
    calls = {"fused": (x, *w, *rope, None), "fused_ex": (x, *w, *rope, *opt),
             "fused_ex_w4": (x, *(t for p in int4 for t in p), *rope, *opt, 128),
             "gemm": (x[0], *int4[0], 128)}
    mqk.fused_qkv_rope_ex(x, *w, *rope, input_norm_w=gam)  # (the workspace)
    mqk.w4a16_gemm(x[0], *int4[0])
    old = sys.getswitchinterval()
    for name, args in calls.items():
        fn, seen, stop = getattr(ext, name), [0], []
        assert type(fn(*args)) in (tuple, torch.Tensor), name
        torch.cuda.synchronize()

        def count():
            while not stop:
                seen[0] += 1
                _native.version()  # (ctypes: gives the GIL up, and must get it again)
        sys.setswitchinterval(1000.0)
        try:
            t = threading.Thread(target=count)
            t.start()
            before = seen[0]
            keep = []
            while seen[0] < before + 20 and len(keep) < 3000:
                keep.append(fn(*args))
            got = seen[0] - before
        finally:
            stop.append(1)
            sys.setswitchinterval(old)
            t.join()
        assert got >= 20, f"{name}: {got} turns of the other thread in {len(keep)} calls"
        torch.cuda.synchronize()
