"""Second branches of a step (a part's work on a stream beside the caller's), on the host alone: streams that only note who waits
for whom, and parts whose kernels are left out."""
import contextlib
import importlib

import pytest
import torch

K = importlib.import_module("daisi-llogos_amd.ops.kernels")
P = importlib.import_module("daisi-llogos_amd.parts")
base = importlib.import_module("daisi-llogos_amd.parts.base")


class Streams:
    """The caller's stream and those that parts make, the current one, and every (waiting, waited for)."""

    def __init__(self, monkeypatch):
        self.caller = self.current = self._stream("caller")
        self.waits = []
        monkeypatch.setattr(torch.cuda, "Stream", lambda device=None: self._stream("side"))
        monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: self.current)
        monkeypatch.setattr(torch.cuda, "stream", self._on)
        for part in (P.ParallelBlock, P.RoutedMoE, P.SideBySide):
            monkeypatch.setattr(part, "_side_streams", {})
            monkeypatch.setattr(part, "side_rows", 64)

    def _stream(self, name):
        waits = self
        return type("Stream", (), {"name": name, "wait_stream": lambda s, other: waits.waits.append((s.name, other.name))})()

    @contextlib.contextmanager
    def _on(self, stream):
        before, self.current = self.current, stream
        try:
            yield
        finally:
            self.current = before


class Rows:
    """What stands for rows on the GPU."""
    shape, device, dtype, is_cuda = (3, 64), torch.device("cuda:0"), torch.bfloat16, True

    def element_size(self):
        return 2


class Quiet(P.Mixer):
    """A mixer or feed-forward that notes the stream it is queued on."""

    def __init__(self, streams):
        self.streams, self.ran = streams, []

    def forward(self, ctx, h, cache=None, **more):
        self.ran.append(self.streams.current.name)
        return h


class QuietNorm(base.Norm):
    def forward(self, x, delta=None, rows=None, write_back=True, lazy=False):
        return x


def _routed(streams, monkeypatch):
    """A mixture with a shared expert large enough for a stream of its own, without its kernels."""
    moe = P.RoutedMoE("m.", 64, 4, 2, 32, shared_intermediate=32)
    moe.shared = Quiet(streams)
    monkeypatch.setattr(P.RoutedMoE, "side_bytes", 0)
    monkeypatch.setattr(importlib.import_module("daisi-llogos_amd.parts.moe"), "_float32", lambda rows: rows)
    weight = type("Weight", (), {"view": lambda self, *a: self})()
    monkeypatch.setattr(K, "moe_router", lambda *a, **k: (None, weight))
    monkeypatch.setattr(K, "moe_route", lambda *a: (None, None, None))
    monkeypatch.setattr(K, "moe_product", lambda *a, **k: None)
    monkeypatch.setattr(K, "moe_combine_weighted", lambda y, where, choice, w, n, h, shared, **k: h)
    moe.rt = P.Runtime(torch.device("cuda:0"), torch.bfloat16)
    return moe


def test_a_branch_does_not_fork_again(monkeypatch):
    """A mixture with a shared expert forks once by itself; as the feed-forward of a block that has forked for it already, not again:
    one fork and one join, and the shared expert runs on the block's second stream."""
    streams = Streams(monkeypatch)
    moe = _routed(streams, monkeypatch)
    moe.forward(None, Rows())
    assert streams.waits == [("side", "caller"), ("caller", "side")] and moe.shared.ran == ["side"]

    streams.waits.clear()
    moe.shared.ran.clear()
    mixer = Quiet(streams)
    block = P.ParallelBlock(QuietNorm(), mixer, moe)
    monkeypatch.setattr(K, "residual_add", lambda x, a: None)
    monkeypatch.setattr(K, "sum_parts", lambda a, bias, dtype: a)
    for ctx in (None, type("Ctx", (), dict(probe=None, n_tokens=3))()):
        block.forward(ctx, Rows(), None, None)
    assert streams.waits == [("side", "caller"), ("caller", "side")] * 2
    assert moe.shared.ran == ["side"] * 2 and mixer.ran == ["caller"] * 2

    with pytest.raises(RuntimeError):                                        # a branch that ends by an error leaves none behind
        monkeypatch.setattr(K, "moe_router", lambda *a, **k: (_ for _ in ()).throw(RuntimeError()))
        block.forward(None, Rows(), None, None)
    streams.waits.clear()
    with pytest.raises(RuntimeError):
        moe.forward(None, Rows())
    assert streams.waits == [("side", "caller")]


def test_branches_that_run_at_the_same_time_share_no_scratch_and_no_counters(monkeypatch):
    """Two attentions side by side: each takes scratch memory and ticket counters of its own, the same ones in every step, launched,
    run before a capture or captured (where none may be made)."""
    streams = Streams(monkeypatch)
    monkeypatch.setattr(P.SideBySide, "side_bytes", 0)
    monkeypatch.setattr(K, "_attn_workspaces", {})
    monkeypatch.setattr(K, "pair_norm", lambda *a, **k: None)
    capturing = []
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: bool(capturing))
    cpu = torch.device("cpu")

    class Attention(Quiet):
        def forward(self, ctx, h, cache=None, **more):
            scratch, counters = K._attn_shares(ctx, cpu, 100, 8)
            self.ran.append((streams.current.name, scratch.data_ptr(), counters.data_ptr(), K._attn_workspace(cpu, 100).data_ptr()))
            return h

    beside = P.SideBySide.__new__(P.SideBySide)
    beside.left, beside.right, beside._left_bytes, beside.norm_w, beside.eps = Attention(streams), Attention(streams), 0, [None, None], 0.0
    ctx = type("Ctx", (), dict(n_tokens=3, probe=None, runtime=P.Runtime(cpu, torch.bfloat16)))()
    rows = torch.zeros(3, 64)
    for step in range(3):
        if step == 2:
            capturing.append(True)
        beside.forward(ctx, rows, [None, None])
    assert [r[0] for r in beside.left.ran] == ["side"] * 3 and [r[0] for r in beside.right.ran] == ["caller"] * 3
    assert len(set(beside.left.ran)) == len(set(beside.right.ran)) == 1
    left, right = beside.left.ran[0][1:], beside.right.ran[0][1:]
    assert len(set(left + right)) == 6


def test_engines_on_one_runtime_share_no_counters():
    """Two engines over one bound model may step at the same time, each on its own stream: what a Runtime holds for an engine's steps is
    that engine's."""
    engine = importlib.import_module("daisi-llogos_amd.engine.step").Engine
    spec = type("Spec", (), dict(max_position=None, vocab_size=8))
    model = type("Model", (), dict(spec=spec, graph_safe=False, cache_needs=lambda self: [], cache_reads=lambda self: []))()
    rt = P.Runtime(torch.device("cpu"), torch.bfloat16)
    first, second = engine(model, rt, 64), engine(model, rt, 64)
    held = [id(getattr(e, name)) for e in (rt, first.rt, second.rt) for name in ("attention_shares", "branch_attention_shares")]
    assert len(set(held)) == 6 and first.rt == rt
