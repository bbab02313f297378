"""The decode kernel's 16- and 32-row blocks against its 64-row block.

A token row's arithmetic does not depend on the block it sits in (the same MFMA
fragments, split order and finish), so a call of T <= 32 tokens must give the bits of
the same rows in a 64-token call, whose kernel is held to the oracle elsewhere; and
the recompute path must give them too.  T at the edges of the blocks; splits of one
tile, of several, of exactly one and of more than one 16-tile slice (where 64 rows and
int4 weights run two slices), at head_dim 128 and 64, with the paged write.
"""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

ROWS = 512


def _case(hidden, Hq, Hkv, D, kind, device):
    g = torch.Generator(device=device).manual_seed(hidden + Hq)
    dt = torch.float16 if kind == "f16" else torch.bfloat16
    rnd = lambda *s: torch.randn(*s, generator=g, device=device)
    x = rnd(64, 1, hidden).to(dt)
    if kind == "w4":
        w = [(torch.randint(-2**31, 2**31 - 1, (hidden // 8, h * D), generator=g, device=device).int(),
              (0.005 + 0.015 * torch.rand(hidden // 64, h * D, generator=g, device=device)).half(),
              torch.randint(-2**31, 2**31 - 1, (hidden // 64, h * D // 8), generator=g, device=device).int())
             for h in (Hq, Hkv, Hkv)]
    else:
        w = [(0.02 * rnd(h * D, hidden)).to(dt) for h in (Hq, Hkv, Hkv)]
    gq, gk = ((1 + 0.1 * rnd(D)).to(dt) for _ in range(2))
    cos, sin = (rnd(ROWS, D).to(dt) for _ in range(2))
    pos = torch.randint(0, ROWS, (64,), generator=g, device=device, dtype=torch.int32)
    return x, w, gq, gk, cos, sin, pos


def _run(case, T, kind):
    import mqk
    x, w, gq, gk, cos, sin, pos = case
    if kind == "w4":
        return mqk.fused_qkv_rope_w4a16(x[:T], *w, gq, gk, cos, sin, pos[:T], group_size=64)
    return mqk.fused_qkv_rope(x[:T], *w, gq, gk, cos, sin, pos[:T])


@pytest.mark.parametrize("kind", ["bf16", "f16", "w4"])
@pytest.mark.parametrize("hidden,Hq,Hkv,D,splits", [
    (64, 2, 1, 128, 0), (1024, 16, 8, 128, 0), (4096, 32, 8, 128, 0), (5120, 40, 8, 128, 0),
    (4096, 32, 8, 128, 16), (2048, 32, 4, 128, 2), (2112, 16, 8, 128, 2), (4096, 8, 4, 128, 2),
    (1024, 16, 8, 64, 0)])
def test_small_blocks_give_the_64_row_bits(hidden, Hq, Hkv, D, splits, kind, device):
    import mqk
    case = _case(hidden, Hq, Hkv, D, kind, device)
    mqk.set_option("decode_splits", splits)
    try:
        want = _run(case, 64, kind)
        for T in (1, 15, 16, 17, 31, 32, 33):
            for recompute in (0, 1) if T in (1, 16, 17, 32) else (0,):
                mqk.set_option("decode_force_recompute", recompute)
                got = _run(case, T, kind)
                mqk.set_option("decode_force_recompute", 0)
                torch.cuda.synchronize()
                for name, a, b in zip("qkv", got, want):
                    assert torch.isfinite(b.float()).all()
                    assert torch.equal(a.view(torch.int16), b[:T].view(torch.int16)), f"T={T} {name} recompute={recompute}"
    finally:
        mqk.set_option("decode_splits", 0)
        mqk.set_option("decode_force_recompute", 0)


@pytest.mark.parametrize("T", [5, 20])
def test_small_blocks_write_the_paged_cache(T, device):
    """K and V rows land in their slots (the returned rows, bit for bit), nothing else
    is written, and a token past the table is skipped."""
    import mqk
    hidden, Hq, Hkv, D = 1024, 16, 8, 128
    x, w, gq, gk, cos, sin, pos = _case(hidden, Hq, Hkv, D, "bf16", device)
    kc, vc = (torch.full((T * 4, 16, Hkv, D), 7.0, dtype=torch.bfloat16, device=device) for _ in range(2))
    table = torch.randperm(T * 4, generator=torch.Generator().manual_seed(T)).int().reshape(T, 4).to(device)
    seq = torch.arange(T, dtype=torch.int32, device=device)
    at = (seq * 7) % 64
    at[T - 1] = 64  # a page past the table
    q, k, v = mqk.fused_qkv_rope_paged(x[:T], *w, gq, gk, cos, sin, kc, vc, table, positions=pos[:T], kv_seq=seq,
                                       kv_pos=at)
    torch.cuda.synchronize()
    want_k, want_v = torch.full_like(kc, 7.0), torch.full_like(vc, 7.0)
    for t in range(T - 1):
        b = int(table[t, int(at[t]) // 16])
        want_k[b, int(at[t]) % 16], want_v[b, int(at[t]) % 16] = k[t, 0], v[t, 0]
    assert torch.equal(kc, want_k) and torch.equal(vc, want_v)
