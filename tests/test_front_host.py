"""What the Python entry points hand to the C++ front, checked with a stand-in for it (no GPU)."""
from __future__ import annotations

import pytest
import torch


class _Front:
    """Takes every call it is given."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def take(*args):
            self.calls.append((name, args))
            return ("taken",)
        return take


@pytest.fixture
def stand_in(monkeypatch):
    from mqk import _native
    f = _Front()
    monkeypatch.setattr(_native, "_front", f)
    return f


def _args(int4):
    t = torch.zeros(1, 2, 256).bfloat16()
    return (t, *([(t, t, t)] * 3 if int4 else [t] * 3), t, t, t, t)


@pytest.mark.parametrize("entry,int4", [("fused_qkv_rope_paged", False), ("fused_qkv_rope_w4a16_paged", True)])
def test_a_paged_call_without_a_cache_is_not_ordinary(entry, int4, stand_in):
    """With k_cache, v_cache and block_table None the paged entry points refuse; the
    extension would take the same arguments as a call that has no cache to write."""
    import mqk
    with pytest.raises(Exception):
        getattr(mqk, entry)(*_args(int4), None, None, None)
    assert stand_in.calls == []
    cache = torch.zeros(1)
    assert getattr(mqk, entry)(*_args(int4), cache, cache, cache) == ("taken",)
