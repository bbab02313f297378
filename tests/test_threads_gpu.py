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
