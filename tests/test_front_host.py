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


def test_an_absent_extension_is_said_once(monkeypatch):
    import sys
    import warnings
    from mqk import _native
    if not _native.LIB_PATH.exists():
        pytest.skip("needs the built library")
    monkeypatch.setattr(_native, "_front", None)
    monkeypatch.setattr(_native, "_front_absent", False)
    monkeypatch.delattr("mqk._front", raising=False)
    monkeypatch.setitem(sys.modules, "mqk._front", None)
    with pytest.warns(RuntimeWarning, match="mqk._front"):
        assert _native.front() is None
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert _native.front() is None


def _build_module():
    import importlib.util
    from pathlib import Path
    path = Path(__file__).resolve().parents[1] / "mini-qwen-llm_amd" / "csrc" / "build.py"
    spec = importlib.util.spec_from_file_location("mqk_csrc_build", path)
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def test_the_library_is_built_without_the_extension(monkeypatch, tmp_path):
    """The C ABI's library needs neither torch nor a host compiler: it is linked (a stand-in
    for the compiler here) also where the extension fails, and the failure is raised after."""
    import subprocess
    from pathlib import Path
    build = _build_module()
    monkeypatch.setattr(build, "BUILD_DIR", tmp_path)
    monkeypatch.setattr(build, "OUT", tmp_path / "libmqk.so")
    monkeypatch.setattr(build, "FRONT", tmp_path / "_front.so")
    monkeypatch.setattr(build, "_hipcc", lambda: "hipcc")
    monkeypatch.setattr(build, "_compile", lambda src, *a: tmp_path / (src + ".o"))

    def run(cmd, **kw):
        if cmd[0] != "hipcc":
            return subprocess.CompletedProcess(cmd, 1, "", "no compiler")
        Path(cmd[cmd.index("-o") + 1]).write_text("linked")
        return subprocess.CompletedProcess(cmd, 0, "", "")
    monkeypatch.setattr(build.subprocess, "run", run)
    build.FRONT.write_text("older")
    with pytest.raises(RuntimeError, match="front.cpp failed"):
        build.build()
    assert build.OUT.read_text() == "linked" and not build.FRONT.exists()
    build.OUT.unlink()
    monkeypatch.setattr(build.importlib.util, "find_spec", lambda name: None)
    assert build.build() == build.OUT and build.OUT.exists()
