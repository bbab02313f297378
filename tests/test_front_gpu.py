"""The C++ form of the entry points (mqk._front) against the Python one.

Both must accept and refuse the same calls and give the same bits: each form below is
run with the extension and with it switched off (``_native._front`` None and marked
absent), and the results, or the exceptions' types and messages, are compared.  Forms:
every entry point and option, the dtypes, head_dim 64 / 96 / 128, odd strides and
offsets, int64 positions, wrong shapes, types and devices, empty calls, subclasses,
autograd inputs, inference mode, torch modes, functorch wrappers, streams and capture.
"""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

H, HQ, HKV, T = 256, 4, 2, 6


class _Sub(torch.Tensor):
    pass


def _base(device, D=128, dt=torch.bfloat16, B=2, S=3, rows=64):
    g = torch.Generator(device=device).manual_seed(D + S)
    r = lambda *s: torch.randn(*s, generator=g, device=device).to(dt)
    return {"x": r(B, S, H), "w_q": 0.05 * r(HQ * D, H), "w_k": 0.05 * r(HKV * D, H), "w_v": 0.05 * r(HKV * D, H),
            "q_norm_w": 1 + 0.1 * r(D), "k_norm_w": 1 + 0.1 * r(D), "cos": r(rows, D), "sin": r(rows, D)}


def _int4(device, N, seed, group=128):
    g = torch.Generator(device=device).manual_seed(seed)
    return (torch.randint(-2**31, 2**31 - 1, (H // 8, N), generator=g, device=device).int(),
            (0.005 + 0.015 * torch.rand(H // group, N, generator=g, device=device)).half(),
            torch.randint(-2**31, 2**31 - 1, (H // group, N // 8), generator=g, device=device).int())


def _offset(t):
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:]
    return flat.copy_(t.reshape(-1)).reshape(t.shape)


def _strided(t):
    return torch.stack([t, t], -1)[..., 0]


def _outcome(fn):
    try:
        out = fn()
        torch.cuda.synchronize()
    except Exception as e:  # noqa: BLE001 (compared below)
        return type(e), str(e)
    out = out if isinstance(out, tuple) else (out,)
    return tuple(None if o is None else o.clone() for o in out)


def _both(fn):
    """Outcomes with the extension and without it (the stream's workspace is warm for both)."""
    from mqk import _native
    assert _native.front() is not None, "mqk._front is built with the library"
    ext = _native._front
    _native._front, _native._front_absent = None, True
    try:
        _outcome(fn)
        general = _outcome(fn)
    finally:
        _native._front, _native._front_absent = ext, False
    return _outcome(fn), general


def _same(fn, label):
    fast, general = _both(fn)
    if general and isinstance(general[0], type):
        assert fast == general, label
        return
    assert not (fast and isinstance(fast[0], type)), f"{label}: {fast}"
    assert len(fast) == len(general), label
    for a, b in zip(fast, general):
        assert (a is None) == (b is None), label
        if a is not None:
            assert type(a) is type(b) and a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride(), label
            assert a.requires_grad == b.requires_grad and a.is_inference() == b.is_inference(), label
            assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8)), label


def _paged(device, D=128, dt=torch.bfloat16):
    kc, vc = (torch.zeros(12, 16, HKV, D, dtype=dt, device=device) for _ in range(2))
    return {"k_cache": kc, "v_cache": vc, "block_table": torch.arange(12, device=device).reshape(6, 2).int()}


def _i(device, *v, dt=torch.int32):
    return torch.tensor(v, dtype=dt, device=device)


def test_plain_forms(device):
    import mqk
    pos = _i(device, 3, 1, 60, 0, 9, 9)
    for D in (64, 96, 128):
        for dt in (torch.bfloat16, torch.float16, torch.float32):
            _same(lambda: mqk.fused_qkv_rope(**_base(device, D, dt)), f"D={D} {dt}")
            _same(lambda: mqk.fused_qkv_rope(**_base(device, D, dt), positions=pos), f"D={D} {dt} positions")
    b = _base(device)
    _same(lambda: mqk.fused_qkv_rope(**b, positions=pos.long()), "int64 positions")
    _same(lambda: mqk.fused_qkv_rope(**b, positions=pos.reshape(2, 3)), "2-D positions")
    _same(lambda: mqk.fused_qkv_rope(**b, positions=pos[:5]), "short positions")
    _same(lambda: mqk.fused_qkv_rope(**b, positions=pos.float()), "float positions")
    _same(lambda: mqk.fused_qkv_rope(**b, positions=[0] * 6), "list positions")
    _same(lambda: mqk.fused_qkv_rope(**b, positions=pos.cpu()), "CPU positions")
    _same(lambda: mqk.fused_qkv_rope(**b, positions=_i(device, -5, 1000, 2, 2**31 - 1, 0, -2**31)), "clamped positions")
    for name in b:
        for how in (_offset, _strided, lambda t: t.half(), lambda t: t.float(), lambda t: t.cpu(), lambda t: t[:1],
                    lambda t: t[..., :64], lambda t: t.reshape(-1), lambda t: t.unsqueeze(0), lambda t: None,
                    lambda t: t.as_subclass(_Sub), lambda t: torch.nn.Parameter(t), lambda t: t.clone().requires_grad_(),
                    lambda t: t[:0], lambda t: t.to(torch.float64), lambda t: t.numpy if False else "tensor"):
            c = dict(b)
            c[name] = how(b[name])
            _same(lambda: mqk.fused_qkv_rope(**c), f"{name} changed")
    _same(lambda: mqk.fused_qkv_rope(**{**b, "x": b["x"].transpose(0, 1)}), "transposed x")
    _same(lambda: mqk.fused_qkv_rope(**{**b, "w_q": b["w_q"].t().contiguous().t()}), "column-major weight")
    _same(lambda: mqk.fused_qkv_rope(**{**b, "x": torch.full_like(b["x"], float("nan"))}), "NaN")


def test_ex_and_paged_forms(device):
    import mqk
    pos = _i(device, 3, 1, 60, 0, 9, 9)
    seq, at = _i(device, 0, 1, 2, 3, 4, 5), _i(device, 0, 31, 5, 16, 7, 40)
    gin = torch.ones(H, device=device).bfloat16() * 1.5
    for D in (64, 96, 128):
        b = _base(device, D)

        def paged(**kw):
            p = _paged(device, D)
            out = mqk.fused_qkv_rope_paged(**b, **p, **kw)
            return (*out, p["k_cache"], p["v_cache"])

        def ex(**kw):
            p = _paged(device, D) if kw.pop("cache", False) else {}
            out = mqk.fused_qkv_rope_ex(**{**b, **kw.pop("base", {})}, **{**p, **kw})
            return (*out, p.get("k_cache"), p.get("v_cache"))
        for kv in (True, False):
            _same(lambda: paged(return_kv=kv), f"paged D={D} {kv}")
            _same(lambda: paged(positions=pos, kv_seq=seq, kv_pos=at, return_kv=kv), f"paged positions D={D} {kv}")
            _same(lambda: ex(cache=True, input_norm_w=gin, positions=pos, kv_seq=seq, kv_pos=at, return_kv=kv), f"ex D={D}")
        _same(lambda: paged(positions=pos), "positions without slots")
        none = {"k_cache": None, "v_cache": None, "block_table": None}
        for kw in (none, {**none, "return_kv": False}, {**none, "positions": pos, "kv_seq": seq, "kv_pos": at},
                   {**_paged(device, D), "k_cache": None}, {**_paged(device, D), "block_table": None}):
            _same(lambda: mqk.fused_qkv_rope_paged(**b, **kw), "paged without a cache")
            assert isinstance(_outcome(lambda: mqk.fused_qkv_rope_paged(**b, **kw))[0], type), "refused"
        _same(lambda: paged(positions=pos, kv_seq=seq.long(), kv_pos=at.long()), "int64 slots")
        _same(ex, "plain ex")
        _same(lambda: ex(return_kv=False), "no cache, no kv")
        _same(lambda: ex(kv_seq=seq), "slots without a cache")
        _same(lambda: ex(cache=True, v_cache=None), "half a cache")
        _same(lambda: ex(cache=True, k_cache=torch.zeros(12, 16, HKV, D, device=device)), "fp32 cache")
        _same(lambda: ex(cache=True, k_cache=torch.zeros(11, 16, HKV, D, device=device).bfloat16()), "cache shapes")
        # (distinct blocks: two tokens that share a slot are written in no defined order)
        _same(lambda: ex(cache=True, block_table=torch.arange(12, device=device).reshape(6, 2)), "int64 table")
        _same(lambda: ex(cache=True, block_table=torch.zeros(12, device=device).int()), "1-D table")
        _same(lambda: ex(input_norm_w=gin, input_eps=1e-5), "norm")
        _same(lambda: ex(input_norm_w=gin, input_eps=1), "integer eps")
        _same(lambda: ex(input_norm_w=gin, input_eps=-1.0), "negative eps")
        _same(lambda: ex(input_norm_w=gin[:64]), "short norm")
        _same(lambda: ex(input_norm_w=gin.float()), "fp32 norm")
        _same(lambda: ex(input_norm_w=_offset(gin)), "unaligned norm")
        cu = _i(device, 0, 2, 6)
        flat = {"x": b["x"].reshape(T, H)}
        _same(lambda: ex(cu_seqlens=cu, base=flat), "varlen")
        _same(lambda: ex(cu_seqlens=cu, seq_pos0=_i(device, 5, 0), cache=True, input_norm_w=gin, base=flat), "varlen all")
        _same(lambda: ex(cu_seqlens=cu), "varlen 3-D")
        _same(lambda: ex(base=flat), "2-D x alone")
        _same(lambda: ex(cu_seqlens=cu, positions=pos), "varlen and positions")
        _same(lambda: ex(seq_pos0=_i(device, 5, 0)), "starts alone")
        _same(lambda: ex(cu_seqlens=cu, seq_pos0=_i(device, 5)), "short starts")
        _same(lambda: ex(cu_seqlens=cu.long(), base=flat), "int64 offsets")
        _same(lambda: ex(cu_seqlens=_i(device, 0)), "one offset")
        _same(lambda: mqk.fused_qkv_rope_varlen(flat["x"], *list(b.values())[1:], cu), "varlen entry")
        _same(lambda: ex(base={"x": b["x"].half()}), "fp16 x")
        _same(lambda: ex(base={"x": b["x"][:, :0]}), "no tokens")


def test_w4a16_forms(device):
    import mqk
    pos = _i(device, 3, 1, 60, 0, 9, 9)
    gin = torch.ones(H, device=device).bfloat16() * 1.5
    for D in (64, 96, 128):
        b = _base(device, D)
        w = [_int4(device, h * D, 7 + i) for i, h in enumerate((HQ, HKV, HKV))]
        rope = (b["q_norm_w"], b["k_norm_w"], b["cos"], b["sin"])
        mods = []
        for t in w:
            m = mqk.LinearW4A16(H, t[0].shape[1], 128, scale_dtype=torch.float16).to(device)
            m.qweight, m.scales, m.qzeros = t
            mods.append(m)
        _same(lambda: mqk.fused_qkv_rope_w4a16(b["x"], *w, *rope), f"tuples D={D}")
        _same(lambda: mqk.fused_qkv_rope_w4a16(b["x"], *mods, *rope, pos), f"modules D={D}")
        _same(lambda: mqk.fused_qkv_rope_w4a16_ex(b["x"], *mods, *rope, pos, input_norm_w=gin), f"norm D={D}")

        def paged():
            p = _paged(device, D)
            out = mqk.fused_qkv_rope_w4a16_paged(b["x"], *mods, *rope, **p)
            return (*out, p["k_cache"], p["v_cache"])
        _same(paged, f"paged D={D}")
        for p in (dict.fromkeys(_paged(device, D)), {**_paged(device, D), "v_cache": None},
                  {**dict.fromkeys(_paged(device, D)), "return_kv": False}):
            call = lambda: mqk.fused_qkv_rope_w4a16_paged(b["x"], *mods, *rope, **p)
            _same(call, "paged without a cache")
            assert isinstance(_outcome(call)[0], type), "refused"
        _same(lambda: mqk.fused_qkv_rope_w4a16(b["x"], *w, *rope, group_size=64), "wrong group")
        _same(lambda: mqk.fused_qkv_rope_w4a16(b["x"], *w, *rope, group_size=0), "group 0")
        _same(lambda: mqk.fused_qkv_rope_w4a16(b["x"], *w, *rope, group_size=True), "boolean group")
        bf = [(q, s.bfloat16(), z) for q, s, z in w]
        _same(lambda: mqk.fused_qkv_rope_w4a16(b["x"], *bf, *rope), "bf16 scales")
        _same(lambda: mqk.fused_qkv_rope_w4a16(b["x"], w[0], bf[1], w[2], *rope), "mixed scales")
        _same(lambda: mqk.fused_qkv_rope_w4a16(b["x"], w[0], w[1], w[0], *rope), "v of q's width")
        _same(lambda: mqk.fused_qkv_rope_w4a16(b["x"], w[0][:2], w[1], w[2], *rope), "two tensors")
        _same(lambda: mqk.fused_qkv_rope_w4a16(b["x"].reshape(T, H), *w, *rope), "2-D x")
        _same(lambda: mqk.fused_qkv_rope_w4a16(b["x"].float(), *w, *rope), "fp32 x")
    x = b["x"].reshape(T, H)
    for arg in ((x, *w[0]), (x[:0], *w[0]), (_strided(x), *w[0]), (_offset(x), *w[0]), (x.float(), *w[0]),
                (x, w[0][0].long(), *w[0][1:]), (x, w[0][0], w[0][1].float(), w[0][2]), (x[:, :128], *w[0]),
                (b["x"], *w[0]), (x.as_subclass(_Sub), *w[0])):
        _same(lambda: mqk.w4a16_gemm(*arg), f"gemm {[tuple(t.shape) for t in arg]}")
    _same(lambda: mqk.w4a16_gemm(x, *w[0], 48), "gemm group 48")
    _same(lambda: mods[0](x), "module 2-D")
    _same(lambda: mods[0](b["x"]), "module 3-D")
    _same(lambda: mods[0](b["x"].reshape(-1)), "module 1-D")


def test_ordinary_calls_are_taken(device):
    """What the fronts are for does go through the extension: each entry point's
    ordinary calls give a result there, not None."""
    import mqk
    from mqk import _native
    ext = _native.front()
    for dt in (torch.bfloat16, torch.float16, torch.float32):
        for D in (64, 128):
            b = list(_base(device, D, dt).values())
            mqk.fused_qkv_rope(*b)  # (the workspace)
            assert type(ext.fused(*b, None)) is tuple, (dt, D)
    b = list(_base(device).values())
    b[1] = torch.nn.Parameter(b[1])
    assert type(ext.fused(*b, _i(device, 0, 1, 2, 3, 4, 5))) is tuple
    p = _paged(device)
    gin = torch.ones(H, device=device).bfloat16()
    opt = (None, None, None, gin, 1e-6, p["k_cache"], p["v_cache"], p["block_table"], None, None)
    mqk.fused_qkv_rope_ex(*b, input_norm_w=gin)
    assert type(ext.fused_ex(*b, *opt, False)) is tuple
    w = [_int4(device, h * 128, 7 + i) for i, h in enumerate((HQ, HKV, HKV))]
    assert type(ext.fused_ex_w4(b[0], *(t for trio in w for t in trio), *b[4:], *opt, True, 128)) is tuple
    assert type(ext.gemm(b[0].reshape(T, H), *w[0], 128)) is torch.Tensor
    assert ext.fused(*[t.cpu() for t in b], None) is None


def test_modes_streams_and_capture(device):
    import mqk
    from mqk import _native
    from torch.utils._python_dispatch import TorchDispatchMode
    b = _base(device)
    call = lambda: mqk.fused_qkv_rope(**b)
    with torch.inference_mode():
        _same(call, "inference mode")

    class Count(TorchDispatchMode):
        n = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            Count.n += 1
            return func(*args, **(kwargs or {}))

    def counted():
        with Count():
            return call()
    _same(counted, "dispatch mode")
    seen = Count.n
    counted()
    assert Count.n > seen  # the outputs are made under the mode
    _same(lambda: torch.vmap(lambda v: mqk.fused_qkv_rope(**{**b, "x": v})[0])(b["x"].unsqueeze(0)), "vmap")
    want = call()
    s = torch.cuda.Stream(device)
    with torch.cuda.stream(s):
        got = [call() for _ in range(3)][-1]
        assert (device.index or 0, int(s.cuda_stream)) in _native._workspaces or \
            _native.fused_workspace_bytes(T, HQ, HKV, H, 128) == 0
        s.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            out = call()
    for _ in range(3):
        for o in out:
            o.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, w) and torch.equal(o, w) for a, o, w in zip(got, out, want))
    # two threads, each on a stream of its own
    import threading
    res = {}

    def work(i):
        st = torch.cuda.Stream(device)
        with torch.cuda.stream(st):
            res[i] = [call() for _ in range(50)][-1]
            st.synchronize()
    th = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    [t.start() for t in th]
    [t.join() for t in th]
    assert all(torch.equal(a, w) for r in res.values() for a, w in zip(r, want))
