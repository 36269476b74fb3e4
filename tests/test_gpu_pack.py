"""trmoe_pack_weight against a torch re-layout, element for element, for every
source order its kernels distinguish: contiguous along K, contiguous along the
output rows, neither; aligned and unaligned starts; sizes around the 128 x 64
tile and the 16-byte vectors."""

import pytest
import torch

from complexity_amd import _native as N
from complexity_amd import ops

pytestmark = pytest.mark.gpu

_DT = {"f32": torch.float32, "bf16": torch.bfloat16, "e4m3": torch.float8_e4m3fn}


def _draw(shape, dtype, gen):
    t = torch.randint(1, 120, shape, generator=gen, dtype=torch.int32)
    if dtype is torch.float8_e4m3fn:
        return t.to(torch.uint8).view(dtype)
    return t.to(dtype)


def _stored(t, order, offset):
    """t [G, O, I] with the same values laid out as `order` asks, `offset` elements into its storage."""
    perm = {"k": (0, 1, 2), "rows": (0, 2, 1), "neither": (1, 2, 0)}[order]
    raw = t.view(torch.uint8) if t.dtype is torch.float8_e4m3fn else t
    p = raw.permute(perm)
    buf = torch.empty(p.numel() + offset, dtype=raw.dtype, device=raw.device)
    v = buf[offset:].view(p.shape)
    v.copy_(p)
    inv = [perm.index(i) for i in range(3)]
    return v.permute(inv), buf


def _expected(a, b, align):
    G, O, I = a.shape
    cols = (I + 7) // 8 * 8
    if b is None:
        rows = (O + align - 1) // align * align
        out = torch.zeros(G, rows, cols, dtype=a.dtype)
        out[:, :O, :I] = a
        return out
    half = align // 2
    feats = (O + half - 1) // half * half
    g, u = torch.zeros(2, G, feats, cols, dtype=a.dtype)
    g[:, :O, :I], u[:, :O, :I] = a, b
    return torch.stack((g.view(G, -1, 32, cols), u.view(G, -1, 32, cols)), 2).reshape(G, 2 * feats, cols)


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("order", ["k", "rows", "neither"])
@pytest.mark.parametrize("dims", [(1, 1, 1), (2, 33, 64), (3, 64, 65), (1, 130, 896), (2, 257, 40), (1, 96, 127)])
@pytest.mark.parametrize("dtype", ["f32", "bf16", "e4m3"])
@pytest.mark.parametrize("gate_up", [True, False])
def test_pack_matches_relayout(gpu, gate_up, dtype, dims, order, offset):
    G, O, I = dims
    gen = torch.Generator().manual_seed(G * 1000 + O + I)
    dt = _DT[dtype]
    a, b = _draw(dims, dt, gen), _draw(dims, dt, gen) if gate_up else None
    raw = (lambda t: t.view(torch.uint8)) if dtype == "e4m3" else (lambda t: t)
    va, keep_a = _stored(a.to(gpu), order, offset)
    vb, keep_b = _stored(b.to(gpu), order, offset) if gate_up else (None, None)
    kw = {}
    if dtype == "e4m3":
        va, vb = va.view(dt), (vb.view(dt) if gate_up else None)
        sa = torch.rand(G, O, generator=gen)
        sb = torch.rand(G, O, generator=gen)
        kw = dict(scale_a=sa.to(gpu), scale_b=sb.to(gpu) if gate_up else None)
    align = 128
    dst, scale = ops._pack(N.PACK_GATE_UP if gate_up else N.PACK_PLAIN, va, vb, G, O, I, va.stride(), align, **kw)
    want = _expected(raw(a), raw(b) if gate_up else None, align)
    assert torch.equal(raw(dst).cpu(), want)
    if dtype == "e4m3":
        ws = _expected(sa[:, :, None], sb[:, :, None] if gate_up else None, align)[:, :, 0]
        assert torch.equal(scale.cpu(), ws)
