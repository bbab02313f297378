"""The fp32 front at the edges of its 16-, 32-, 48- and 64-row tiles and of its k stages.

Against the projection, per-head RMSNorm and RoPE in float64.  Bound: a sum of K fp32
products, every partial sum rounded, is within K * 2^-24 * sum|x w| of the exact
one; the norm and RoPE scale that by |gamma| / rms and add a few ulps of the output.  Row
by row that is far above what is seen (rounding errors average out), so the bar is the
same with sqrt(K) in place of K and a factor of 4 for the tail of ~1e6 samples.
"""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _exact(x, ws, gq, gk, cos, sin, rows, D):
    out, slack = [], []
    for w, g in zip(ws, (gq, gk, None)):
        y = (x.double() @ w.double().T).reshape(len(x), -1, D)
        e = (x.double().abs() @ w.double().abs().T).reshape(len(x), -1, D) * (4 * x.shape[1] ** 0.5 * 2.0 ** -24)
        if g is not None:
            r = torch.rsqrt((y * y).mean(-1, keepdim=True) + 1e-6)
            # an error of the row moves its rms too: at most its own relative size again
            e = (e + y.abs() * (e.amax(-1, keepdim=True) * r)) * r * g.double().abs()
            y = y * r * g.double()
            c, s = cos.double()[rows][:, None], sin.double()[rows][:, None]
            half = D // 2
            rot = lambda t: torch.cat([-t[..., half:], t[..., :half]], -1)  # noqa: E731
            e = e * c.abs() + torch.cat([e[..., half:], e[..., :half]], -1) * s.abs()
            y = y * c + rot(y) * s
        out.append(y)
        slack.append(e + y.abs() * 2.0 ** -21)
    return out, slack


@pytest.mark.parametrize("T,hidden,Hq,Hkv,D", [
    # k: less than one stage, one, one and a half, two, five and a half, nine and a half stages
    (1, 32, 2, 1, 128), (17, 64, 2, 1, 128), (16, 96, 1, 1, 128), (15, 128, 2, 2, 64), (33, 352, 16, 8, 128),
    (128, 608, 16, 8, 128), (100, 1024, 16, 8, 64),
    # 32, 48 and 64 rows per tile, whole and ragged
    (200, 32, 16, 8, 128), (256, 64, 16, 8, 128), (193, 96, 16, 8, 64), (225, 224, 16, 8, 128), (250, 1056, 16, 8, 128),
    (300, 32, 16, 8, 128), (289, 160, 16, 8, 128), (384, 128, 16, 8, 64), (333, 320, 16, 8, 128),
    (500, 32, 16, 8, 128), (512, 64, 16, 8, 128), (449, 288, 16, 8, 128), (1029, 192, 32, 4, 128),
])
def test_f32_rows_and_stages(T, hidden, Hq, Hkv, D, device):
    import mqk
    g = torch.Generator().manual_seed(1000 * T + hidden)
    x = torch.randn(1, T, hidden, generator=g)
    ws = [torch.randn(h * D, hidden, generator=g) * 0.05 for h in (Hq, Hkv, Hkv)]
    gq, gk = (1 + 0.1 * torch.randn(D, generator=g) for _ in range(2))
    cos, sin = torch.randn(T + 9, D, generator=g), torch.randn(T + 9, D, generator=g)
    pos = torch.randint(0, T + 9, (T,), generator=g, dtype=torch.int32)
    for positions in (None, pos):
        shape = (1, T) if positions is None else (T, 1)
        out = mqk.fused_qkv_rope(*(a.to(device) for a in [x.reshape(*shape, hidden), *ws, gq, gk, cos, sin]),
                                 positions=None if positions is None else positions.to(device))
        torch.cuda.synchronize()
        rows = torch.arange(T) if positions is None else pos.long()
        for name, o, r, e in zip("qkv", out, *_exact(x[0], ws, gq, gk, cos, sin, rows, D)):
            over = ((o.double().cpu().reshape(r.shape) - r).abs() / e).max().item()
            assert over <= 1, f"{name} T={T} hidden={hidden}: {over:.2f} of the bound"
