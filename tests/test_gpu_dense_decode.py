"""The fused decode call against the separate gate|up and down calls it stands
for: the same kernels and sums in the same order, so the outputs are equal bit
for bit, over token counts at the tile and split edges, both dtypes, and
repeated calls (the split counters are cleared by each)."""

import pytest
import torch

from complexity_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,S,E,W", [(896, 3072, 4, 64), (200, 100, 2, 40), (72, 0, 4, 32), (2048, 1500, 2, 64)])
@pytest.mark.parametrize("n", [1, 8, 9, 16, 17, 33, 64, 65, 128])
def test_fused_equals_separate(gpu, n, H, S, E, W, dtype):
    g = torch.Generator().manual_seed(n + H)
    dev = lambda *s: (torch.randn(*s, generator=g) * 0.05).to(gpu).to(dtype)  # noqa: E731
    x, res = dev(n, H) * 20, dev(n, H) * 20
    shared = (dev(S, H), dev(S, H), dev(H, S)) if S else (None, None, None)
    experts = (dev(E, H, W), dev(E, H, W), dev(E, W, H))
    gu, dn, F = ops.pack_dense_routed(*shared, *experts)
    p = ops.PackedLayer(act_dtype=dtype, num_experts=E, expert_width=W, strategy=ops.STRATEGY_DENSE, shared_width=S,
                        dense_gate_up=gu, dense_down=dn, dense_features=F)
    ids = torch.randint(0, 50, (n,), generator=g).to(gpu)
    table = torch.stack((torch.arange(50) % E, (torch.arange(50) + 1) % E)).to(gpu)
    rs = (torch.rand(n, generator=g) + 0.5).to(gpu)
    x = ops.rows16(x)
    for kw in ({}, {"rms_eps": 1e-6}, {"row_scale": rs}):
        h = ops.dense_routed_gate_up(x, gu, S, E, W, ids, table, (0.4, 0.6), 0.75, 2.0,
                                     w_frag=p.fragments("dense_gate_up", H), **kw)
        want = ops.shared_down_combine(h, F, dn, None, H, None, None, 2, (0.4, 0.6), 1.0, 1.0, res,
                                       w_frag=p.fragments("dense_down", F))
        for _ in range(3):
            got = ops.dense_decode(x, ids, table, p, (0.4, 0.6), 0.75, 2.0, res, **kw)
            assert torch.equal(got, want)
