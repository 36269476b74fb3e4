"""The decoder's attention kernels against fp32 torch: q/k norm + rotation +
cache writes, a prompt's causal attention at lengths around the 64-position
tiles and the 128-query workgroups, and one decode step's attention at cache
lengths around the 256-position splits, positions at both ends, and every
supported group size.

Bounds: the kernels round only their bf16 outputs (half a step, 2^-9, of the
value), and the decode attention reads k and v rounded to bf16 as the caches
hold them, which the reference does as well; the projection's inputs x * w are
rounded to bf16 once more (2^-9 each, averaging out over the row).  2^-7 of the
row norm covers both with a factor of two."""

import math

import pytest
import torch
import torch.nn.functional as F

from complexity_amd import ops
from complexity_amd.decoder import rope_tables

pytestmark = pytest.mark.gpu
D = 64


def _rms(x, w, eps=1e-6):
    x = x.float()
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w.float()


def _rope(x, cos, sin):
    return x * cos + torch.cat((-x[..., 32:], x[..., :32]), -1) * sin


def _rel(got, want):
    return float(((got.float() - want).norm(dim=-1) / want.norm(dim=-1)).max())


@pytest.mark.parametrize("B,T,heads,kvh,first,L", [(1, 1, 14, 2, 0, 64), (2, 37, 14, 2, 5, 64), (3, 65, 4, 4, 0, 128),
                                                   (8, 256, 8, 1, 0, 256)])
def test_qk_norm_rope(gpu, B, T, heads, kvh, first, L):
    g = torch.Generator().manual_seed(T)
    kqv = torch.randn(B * T, (heads + 2 * kvh) * D, generator=g).to(gpu).bfloat16()
    qw, kw = ((torch.rand(D, generator=g) + 0.5).to(gpu).bfloat16() for _ in range(2))
    cos, sin = (t.to(gpu) for t in rope_tables(D, L, 10000.0))
    kc, vc = (torch.full((B, kvh, L, D), 7.0, device=gpu, dtype=torch.bfloat16) for _ in range(2))
    pos = torch.tensor([first], device=gpu) if T == 1 else None
    q = ops.qk_norm_rope(kqv, B, heads, qw, kw, 1e-6, cos, sin, kc, vc, 0 if T == 1 else first, pos)
    k, qr, v = kqv.view(B, T, -1, D).split([kvh, heads, kvh], 2)
    c, s = cos[first:first + T, None], sin[first:first + T, None]
    assert _rel(q, _rope(_rms(qr, qw), c, s)) <= 2.0 ** -7
    span = slice(first, first + T)
    assert _rel(kc[:, :, span], _rope(_rms(k, kw), c, s).transpose(1, 2)) <= 2.0 ** -7
    assert torch.equal(vc[:, :, span], v.transpose(1, 2))
    rest = torch.ones(L, dtype=torch.bool)
    rest[span] = False
    assert bool((kc[:, :, rest.to(gpu)] == 7.0).all()) and bool((vc[:, :, rest.to(gpu)] == 7.0).all())


@pytest.mark.parametrize("B,hidden,heads,kvh,L,pos", [
    (1, 896, 14, 2, 64, 0), (1, 896, 14, 2, 2048, 2047), (2, 896, 14, 2, 128, 127), (3, 32, 2, 2, 192, 128),
    (5, 96, 2, 1, 320, 129), (8, 896, 14, 2, 1088, 1000), (9, 544, 8, 1, 256, 255), (16, 64, 16, 4, 4096, 3001)])
def test_decode_attention(gpu, B, hidden, heads, kvh, L, pos):
    g = torch.Generator().manual_seed(pos + B)
    n = (heads + 2 * kvh) * D
    x = torch.randn(B, hidden, generator=g).to(gpu).bfloat16()
    nw = (torch.rand(hidden, generator=g) + 0.5).to(gpu).bfloat16()
    w = (torch.randn(n, hidden, generator=g) * hidden ** -0.5).to(gpu).bfloat16()
    qw, kw = ((torch.rand(D, generator=g) + 0.5).to(gpu).bfloat16() for _ in range(2))
    cos, sin = (t.to(gpu) for t in rope_tables(D, L, 10000.0))
    kc, vc = (torch.randn(B, kvh, L, D, generator=g).to(gpu).bfloat16() for _ in range(2))
    kc[:, :, pos + 1:] = float("nan")   # positions ahead are never read
    position = torch.tensor([pos], device=gpu)
    scale = 1.0 / math.sqrt(D)
    for _ in range(3):   # the split counters are cleared again by every call
        got = ops.decode_attention(x, nw, 1e-6, w, heads, qw, kw, 1e-6, cos, sin, position, kc, vc, scale)
    qkv = _rms(x, nw) @ w.float().t()
    k, q, v = qkv.view(B, -1, D).split([kvh, heads, kvh], 1)
    c, s = cos[pos], sin[pos]
    q, k = _rope(_rms(q, qw), c, s), _rope(_rms(k, kw), c, s)
    assert _rel(kc[:, :, pos], k) <= 2.0 ** -7 and _rel(vc[:, :, pos], v) <= 2.0 ** -7
    keys = kc[:, :, :pos + 1].float().repeat_interleave(heads // kvh, 1)
    vals = vc[:, :, :pos + 1].float().repeat_interleave(heads // kvh, 1)
    p = torch.softmax((keys @ q.unsqueeze(-1)).squeeze(-1) * scale, -1)
    want = (p.unsqueeze(-1) * vals).sum(2)
    assert _rel(got.view(B, heads, D), want) <= 2.0 ** -6   # q's own error moves the weights of up to L positions


@pytest.mark.parametrize("B,T,heads,kvh", [(1, 1, 14, 2), (2, 31, 4, 4), (1, 64, 14, 2), (3, 65, 8, 1), (1, 128, 2, 1),
                                           (1, 197, 14, 2), (2, 300, 3, 1), (1, 2048, 14, 2)])
def test_prefill_attention(gpu, B, T, heads, kvh):
    g = torch.Generator().manual_seed(T)
    L = (T + 63) // 64 * 64 + 64
    q = torch.randn(B, T, heads, D, generator=g).to(gpu).bfloat16() * 2
    kc, vc = (torch.randn(B, kvh, L, D, generator=g).to(gpu).bfloat16() for _ in range(2))
    kc[:, :, T:] = float("nan")   # positions past the prompt are never read
    vc[:, :, T:] = float("nan")
    scale = 1.0 / math.sqrt(D)
    got = ops.prefill_attention(q, kc, vc, scale)
    k, v = (c[:, :, :T].float().repeat_interleave(heads // kvh, 1) for c in (kc, vc))
    s = (q.float().transpose(1, 2) @ k.transpose(2, 3)) * scale
    s.masked_fill_(torch.ones(T, T, dtype=torch.bool, device=gpu).triu(1), -math.inf)
    want = (torch.softmax(s, -1) @ v).transpose(1, 2)
    # the weights are rounded to bf16 (2^-9 each) before the second product
    assert _rel(got.view(B, T, heads, D), want) <= 2.0 ** -7


@pytest.mark.parametrize("rise", [0.01, 0.05, 0.5, -0.5])
def test_prefill_attention_moving_maximum(gpu, rise):
    # scores that climb (or fall) with the position by `rise` a step: the
    # reference point of the exponentials stays for a while, moves at every
    # tile, or never again
    T, L = 700, 768
    q = torch.zeros(1, T, 2, D, device=gpu).bfloat16()
    q[..., 0], q[..., 1] = 8.0, 8.0
    kc = torch.zeros(1, 1, L, D, device=gpu).bfloat16()
    ramp = rise * torch.arange(L, device=gpu)
    kc[..., 0] = ramp.bfloat16()
    kc[..., 1] = (ramp - ramp.bfloat16().float()).bfloat16()   # the ramp to 16 bits
    vc = torch.randn(1, 1, L, D, generator=torch.Generator().manual_seed(1)).to(gpu).bfloat16()
    got = ops.prefill_attention(q, kc, vc, 0.125)
    k, v = (c[:, :, :T].float().expand(1, 2, T, D) for c in (kc, vc))
    s = (q.float().transpose(1, 2) @ k.transpose(2, 3)) * 0.125
    s.masked_fill_(torch.ones(T, T, dtype=torch.bool, device=gpu).triu(1), -math.inf)
    want = (torch.softmax(s, -1) @ v).transpose(1, 2)
    assert _rel(got.view(1, T, 2, D), want) <= 2.0 ** -7


def test_decode_linear_adds_residual(gpu):
    g = torch.Generator().manual_seed(0)
    for n in (1, 8, 9, 16):
        x = torch.randn(n, 896, generator=g).to(gpu).bfloat16()
        w = (torch.randn(896, 896, generator=g) * 0.03).to(gpu).bfloat16()
        r = torch.randn(n, 896, generator=g).to(gpu).bfloat16()
        assert _rel(ops.decode_linear(x, w, r), F.linear(x.float(), w.float()) + r.float()) <= 2.0 ** -8


def test_prefill_attention_of_many_prompts(gpu):
    # more (prompt, head) pairs than 65535: the first, middle and last prompts
    B, T, heads, kvh, L = 4700, 3, 14, 2, 64
    g = torch.Generator(device=gpu).manual_seed(0)
    q = torch.randn(B, T, heads, D, generator=g, device=gpu).bfloat16()
    kc, vc = (torch.randn(B, kvh, L, D, generator=g, device=gpu).bfloat16() for _ in range(2))
    got = ops.prefill_attention(q, kc, vc, 0.125).view(B, T, heads, D)
    for b in (0, 2340, 4680, 4681, 4699):
        assert torch.equal(got[b], ops.prefill_attention(q[b:b + 1], kc[b:b + 1], vc[b:b + 1], 0.125).view(T, heads, D))
