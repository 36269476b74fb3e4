"""Which kernels a decode-sized layer call reaches, on the CPU: the kernel
calls of ops.layer_forward are replaced by recorders."""

import threading
import time

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
def stream(monkeypatch):
    """The current stream: whether it records a graph, and what is done on it."""
    class Stream:
        capturing = False

        def synchronize(self):
            self.did.append("synchronize")

    s = Stream()
    s.did = []
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: s.capturing)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: s)
    monkeypatch.setattr(ops, "pack_e4m3_decode", lambda p, h: s.did.append("pack") or ops.E4M3Decode(*[None] * 4))
    monkeypatch.setattr(ops, "pack_fragments", lambda w, c: s.did.append("pack") or (torch.zeros(1), c))
    return s


@pytest.fixture()
def calls(monkeypatch, stream):
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


def _dense(dtype=BF):
    z = lambda *s: torch.zeros(*s, dtype=dtype)  # noqa: E731
    return ops.PackedLayer(act_dtype=dtype, num_experts=E, expert_width=W, strategy=ops.STRATEGY_DENSE, shared_width=S,
                           dense_gate_up=z(2 * 384, H), dense_down=z(256, 384), dense_features=384)


def test_a_recording_graph_builds_no_e4m3_copy(calls, stream):
    p = _pack()
    stream.capturing = True
    _forward(p)
    assert stream.did == [] and p.e4m3_frag is None and calls[0] == "route_sort"
    stream.capturing = False
    _forward(p)
    assert stream.did == ["pack", "synchronize"] and calls[-1] == "e4m3_decode_layer"
    stream.capturing = True
    _forward(p)   # the copy is there, complete: the graph may read it
    assert stream.did == ["pack", "synchronize"] and calls[-1] == "e4m3_decode_layer"


def test_a_recording_graph_builds_no_fragments(calls, stream, monkeypatch):
    monkeypatch.setattr(ops, "dense_routed_gate_up", lambda *a, **k: calls.append("gate_up") or torch.zeros(3, 384))
    monkeypatch.setattr(ops, "dense_decode", lambda *a, **k: calls.append("fused"))
    p = _dense()
    stream.capturing = True
    _forward(p)
    assert stream.did == [] and p.frag == {} and calls == ["gate_up", "shared_down_combine"]
    stream.capturing = False
    _forward(p)
    assert stream.did == ["pack", "synchronize"] * 2 and calls[-1] == "fused"
    stream.capturing = True
    _forward(p)
    assert len(stream.did) == 4 and calls[-1] == "fused"


def test_a_copy_is_built_once_by_several_threads(stream, monkeypatch):
    made, gate = [], threading.Barrier(8)
    monkeypatch.setattr(ops, "pack_e4m3_decode", lambda p, h: (time.sleep(0.02), made.append(object()), made[-1])[-1])
    p, got = _pack(), []
    ts = [threading.Thread(target=lambda: (gate.wait(), got.append(p.e4m3_decode(H)))) for _ in range(8)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert len(made) == 1 and all(g is made[0] for g in got)


def test_copies_built_together_are_waited_for_once(stream):
    a, b = _dense(), _dense()
    with ops.decode_copies_together():
        got = [p.fragments(n, H) for p in (a, b) for n in ("dense_gate_up", "dense_down")]
        assert stream.did == ["pack"] * 4 and a.frag == b.frag == {}   # no other call finds them yet
        with ops.decode_copies_together():
            pass
        assert a.frag == {}
    assert stream.did == ["pack"] * 4 + ["synchronize"]
    assert got == [p.frag[n] for p in (a, b) for n in ("dense_gate_up", "dense_down")]
    with ops.decode_copies_together():
        assert a.fragments("dense_down", H) is got[1]
    assert len(stream.did) == 5


def test_copies_of_a_failed_batch_are_kept_complete(stream):
    p = _dense()
    with pytest.raises(KeyError):
        with ops.decode_copies_together():
            p.fragments("dense_down", H)
            raise KeyError
    assert stream.did == ["pack", "synchronize"] and list(p.frag) == ["dense_down"]
    p.fragments("dense_gate_up", H)   # alone again
    assert stream.did == ["pack", "synchronize"] * 2
