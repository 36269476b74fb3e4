"""Decode-sized calls of e4m3 layers (one gate|up and one down over the shared
and every expert's features) against the same formula in torch: token counts at
the edges of the 16-row tiles, widths that pad, experts no token reaches (their
weights are skipped), slots naming one expert twice.

The reference rounds h to bf16 where the kernel does, so the two differ by fp32
summation order, the h values that rounding then sends the other way, and the
output's own rounding: within one bf16 step (2^-8) of the row's norm."""

import pytest
import torch
import torch.nn.functional as F

from complexity_amd import ops
from complexity_amd.tr_hash import TRHashEngine, TRHashEngineConfig

pytestmark = pytest.mark.gpu

SHAPES = {
    # hidden, shared, experts, width, top_k
    "scaled": (2048, 5632, 16, 256, 2),
    "padded": (200, 100, 4, 48, 2),
    "no_shared": (256, 0, 8, 64, 4),
    "narrow": (72, 130, 2, 40, 1),
}


def _engine(shape, gpu):
    H, S, E, W, k = SHAPES[shape]
    torch.manual_seed(7)
    cfg = TRHashEngineConfig(hidden_size=H, vocab_size=500, num_experts=E, top_k=k, shared_width=S, expert_width=W,
                             routing_strategy="token_id_multi_hash" if k == 2 else "token_id_balanced_hash", precision="fp8",
                             phase="inference", routed_output_scale=2.0, shared_output_scale=0.75,
                             initializer_range=0.05)
    e = TRHashEngine(cfg).to(device=gpu, dtype=torch.bfloat16)
    e.quantize_fp8_()
    return e.eval()


def _reference(e, x, ids, residual):
    """fp32 on the dequantised weights; h (with its scale and route weight) rounded to bf16."""
    c = e.config
    w = {n: (getattr(e, n + "_fp8").float() * getattr(e, n + "_scale").float().unsqueeze(1))
         for n in ("expert_gate", "expert_up", "expert_down")}
    x = x.float()
    out = torch.zeros_like(x)
    if c.shared_width:
        s = {n: getattr(e, n + "_fp8").float() * getattr(e, n + "_scale").float().unsqueeze(1)
             for n in ("shared_gate", "shared_up", "shared_down")}
        h = F.silu(x @ s["shared_gate"].t()) * (x @ s["shared_up"].t()) * c.shared_output_scale
        out = out + h.bfloat16().float() @ s["shared_down"].t()
    routes = e.route_table[:, ids.reshape(-1)]
    for ex in range(c.num_experts):
        tw = sum((routes[j] == ex).float() * c.route_weights[j] for j in range(c.top_k)) * c.routed_output_scale
        h = F.silu(x @ w["expert_gate"][ex]) * (x @ w["expert_up"][ex]) * tw[:, None]
        out = out + h.bfloat16().float() @ w["expert_down"][ex]
    return out if residual is None else out + residual.float()


@pytest.mark.parametrize("tokens", [1, 3, 4, 5, 8, 9, 16, 17, 32, 33, 64, 65, 128])
@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_decode_matches_formula(gpu, shape, tokens):
    e = _engine(shape, gpu)
    g = torch.Generator().manual_seed(tokens)
    H = e.config.hidden_size
    x = torch.randn(tokens, 1, H, generator=g).to(gpu).bfloat16()
    ids = torch.randint(0, 500, (tokens, 1), generator=g).to(gpu)
    res = torch.randn(tokens, 1, H, generator=g).to(gpu).bfloat16() if tokens % 2 else None
    if tokens == 4:   # both slots of every token on one expert
        e.route_table.zero_()
    with torch.no_grad():
        out = e(x, ids) if res is None else e.forward_with_residual(x, ids, res)
        ref = _reference(e, x.view(-1, H), ids, None if res is None else res.view(-1, H))
    assert e._packed.e4m3_frag is not None
    err = (out.view(-1, H).float() - ref).norm(dim=1) / ref.norm(dim=1)
    assert float(err.max()) <= 2.0 ** -8, float(err.max())


def test_unrouted_overflow_stays_out(gpu):
    """An expert whose SwiGLU overflows leaves the tokens that are not routed to it alone."""
    e = _engine("padded", gpu)
    with torch.no_grad():
        e.expert_gate_scale[0] = e.expert_up_scale[0] = 3e38
    e.load_route_table(torch.tensor([[0] * 250 + [1] * 250, [1] * 250 + [2] * 250]))
    x = torch.ones(40, 1, 200, device=gpu, dtype=torch.bfloat16)
    ids = torch.arange(0, 400, 10, device=gpu).view(40, 1)
    with torch.no_grad():
        out = e(x, ids).float().view(40, -1)
    assert not torch.isfinite(out[:25]).all()
    assert torch.isfinite(out[25:]).all()


def test_graph_recorded_before_any_decode(gpu):
    """A decode call recorded after prompts alone, without a warm-up: eager calls
    before the first replay, between replays and after the graph is gone give
    what they gave without it, and so does every replay."""
    shape, n = "scaled", 32
    g = torch.Generator().manual_seed(0)
    H = SHAPES[shape][0]
    x = torch.randn(n, 1, H, generator=g).to(gpu).bfloat16()
    ids = torch.randint(0, 500, (n, 1), generator=g).to(gpu)
    e, other = _engine(shape, gpu), _engine(shape, gpu)
    other.load_state_dict(e.state_dict())
    with torch.no_grad():
        prompt = torch.randn(1, 300, H, generator=g).to(gpu).bfloat16()
        e(prompt, torch.zeros(1, 300, dtype=torch.int64, device=gpu))
        scope = ops.workspace_scope()
        graph = torch.cuda.CUDAGraph()
        with scope, torch.cuda.graph(graph):
            recorded = e(x, ids)
        want = other(x, ids)          # fused, its copy built eagerly
        ref = _reference(e, x.view(-1, H), ids, None)
        assert torch.equal(e(x, ids), want)
        for _ in range(3):
            graph.replay()
            assert torch.equal(e(x, ids), want)
            # the grouped kernels round the experts' outputs to bf16 once more than the fused ones: 2^-8 each
            err = (recorded.view(-1, H).float() - ref).norm(dim=1) / ref.norm(dim=1)
            assert float(err.max()) <= 2.0 ** -7
        del graph, recorded
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        assert torch.equal(e(x, ids), want)
