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
