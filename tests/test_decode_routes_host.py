"""Which kernels a decode-sized layer call reaches, on the CPU: the kernel
calls of ops.layer_forward are replaced by recorders."""

import pytest
import torch

from complexity_amd import ops

H, S, E, W = 64, 128, 4, 64


def _pack(shared=torch.float8_e4m3fn, experts=torch.float8_e4m3fn, shared_width=S):
    t = lambda d, *s: torch.zeros(*s).to(d)  # noqa: E731
    sc = lambda d, *s: torch.ones(*s) if d is torch.float8_e4m3fn else None  # noqa: E731
    return ops.PackedLayer(
        act_dtype=torch.bfloat16, num_experts=E, expert_width=W, strategy=ops.STRATEGY_GROUPED,
        expert_gate_up=t(experts, E, 2 * W, H), expert_gate_up_scale=sc(experts, E, 2 * W),
        expert_down=t(experts, E, 256, W), expert_down_scale=sc(experts, E, 256), shared_width=shared_width,
        shared_gate_up=t(shared, 2 * S, H) if shared_width else None, shared_gate_up_scale=sc(shared, 2 * S),
        shared_down=t(shared, 256, S) if shared_width else None, shared_down_scale=sc(shared, 256))


@pytest.fixture()
def calls(monkeypatch):
    got = []

    def record(name, out):
        def fn(*a, **kw):
            got.append(name)
            return out() if out else None
        monkeypatch.setattr(ops, name, fn)

    record("e4m3_decode_layer", lambda: torch.zeros(3, H))
    record("route_sort", lambda: (None, None, None, None))
    record("routed_experts", lambda: torch.zeros(6, H))
    record("shared_gate_up", lambda: torch.zeros(3, S))
    record("shared_down_combine", lambda: torch.zeros(3, H))
    record("combine", lambda: torch.zeros(3, H))
    record("pack_fragments", lambda: (torch.zeros(1), 1))
    return got


def _forward(p):
    x = torch.zeros(3, H, dtype=torch.bfloat16)
    ops.layer_forward(x, torch.zeros(3, dtype=torch.int64), torch.zeros(2, 10, dtype=torch.int64), p, (0.5, 0.5), 1.0, 1.0)


F8, BF = torch.float8_e4m3fn, torch.bfloat16


@pytest.mark.parametrize("shared,experts,width,fused", [(F8, F8, S, True), (F8, F8, 0, True), (BF, F8, S, False),
                                                        (F8, BF, S, False), (BF, BF, S, False)])
def test_only_layers_wholly_in_e4m3_take_the_fused_decode(calls, shared, experts, width, fused):
    _forward(_pack(shared, experts, width))
    assert ("e4m3_decode_layer" in calls) == fused and ("route_sort" in calls) == (not fused)
