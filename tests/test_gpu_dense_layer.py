"""The fused dense-routed prefill call against the separate calls, token counts
on both sides of the in-kernel RMSNorm's limit: where the scales come from
trmoe_rms_row_scale the outputs are equal bit for bit; where the gate|up sums
its rows' squares itself, in another order, each scale is off by at most 2^-20
relative and an h value may round the other way, so the outputs agree within
the bf16 (2^-8) or fp32 (2^-18) bound of the layer."""

import pytest
import torch

from complexity_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,S,E,W", [(896, 3072, 4, 64), (200, 100, 2, 40)])
@pytest.mark.parametrize("n", [129, 512, 777, 1100, 1153, 2050])
def test_fused_equals_separate(gpu, n, H, S, E, W, dtype):
    g = torch.Generator().manual_seed(n + H)
    dev = lambda *s: (torch.randn(*s, generator=g) * 0.05).to(gpu).to(dtype)  # noqa: E731
    x = dev(n, H) * torch.logspace(-2, 2, n).to(gpu)[:, None].to(dtype)
    gu, dn, F = ops.pack_dense_routed(dev(S, H), dev(S, H), dev(H, S), dev(E, H, W), dev(E, H, W), dev(E, W, H))
    p = ops.PackedLayer(act_dtype=dtype, num_experts=E, expert_width=W, strategy=ops.STRATEGY_DENSE, shared_width=S,
                        dense_gate_up=gu, dense_down=dn, dense_features=F)
    ids = torch.randint(0, 50, (n,), generator=g).to(gpu)
    table = torch.stack((torch.arange(50) % E, (torch.arange(50) + 1) % E)).to(gpu)
    x = ops.rows16(x)
    h = ops.dense_routed_gate_up(x, gu, S, E, W, ids, table, (0.4, 0.6), 0.75, 2.0, row_scale=ops.rms_row_scale(x, 1e-6))
    want = ops.shared_down_combine(h, F, dn, None, H, None, None, 2, (0.4, 0.6), 1.0, 1.0, None)
    got = ops.dense_layer(x, ids, table, p, (0.4, 0.6), 0.75, 2.0, None, 1e-6)
    rel = float(((got - want).float().norm(dim=1) / want.float().norm(dim=1)).max())
    assert rel <= (2.0 ** -8 if dtype is torch.bfloat16 else 2.0 ** -18), rel
    if dtype is torch.bfloat16 and n > 1152 and H == 896:
        assert torch.equal(got, want)


@pytest.mark.parametrize("H,S,E,W", [(896, 3072, 4, 64), (200, 100, 2, 40)])
@pytest.mark.parametrize("n", [65, 100, 128])
@pytest.mark.parametrize("eps", [None, 1e-6])
def test_above_the_decode_kernels(gpu, n, H, S, E, W, eps):
    # bf16 layers of 65..128 tokens run on tiles; the decode kernels (the separate
    # calls) sum the same products in another order.  h (bf16, rounded to 2^-9
    # relative) may round the other way, and so may the output: 2^-8 of the rows
    g = torch.Generator().manual_seed(n + H)
    dev = lambda *s: (torch.randn(*s, generator=g) * 0.05).to(gpu).bfloat16()  # noqa: E731
    x, res = ops.rows16(dev(n, H) * 20), dev(n, H) * 20
    gu, dn, F = ops.pack_dense_routed(dev(S, H), dev(S, H), dev(H, S), dev(E, H, W), dev(E, H, W), dev(E, W, H))
    p = ops.PackedLayer(act_dtype=torch.bfloat16, num_experts=E, expert_width=W, strategy=ops.STRATEGY_DENSE,
                        shared_width=S, dense_gate_up=gu, dense_down=dn, dense_features=F)
    ids = torch.randint(0, 50, (n,), generator=g).to(gpu)
    table = torch.stack((torch.arange(50) % E, (torch.arange(50) + 1) % E)).to(gpu)
    h = ops.dense_routed_gate_up(x, gu, S, E, W, ids, table, (0.4, 0.6), 0.75, 2.0, rms_eps=eps or 0.0)
    want = ops.shared_down_combine(h, F, dn, None, H, None, None, 2, (0.4, 0.6), 1.0, 1.0, res)
    got = ops.layer_forward(x, ids, table, p, (0.4, 0.6), 0.75, 2.0, residual=res, norm_eps=eps)
    rel = float(((got - want).float().norm(dim=1) / want.float().norm(dim=1)).max())
    assert rel <= 2.0 ** -8, rel
