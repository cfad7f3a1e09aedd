"""The sampler's staging buffers outlive their samplers until their copies have run.  Events and pinned memory are stand-ins here."""
import gc
import importlib
import sys
import threading
import time
import weakref

import pytest
import torch

S = importlib.import_module("daisi-llogos_amd.sampling")
staging = importlib.import_module("daisi-llogos_amd.sampling.sampler")


class Event:
    """A copy's event: not done until the test says so; `asked` runs while it is being asked."""
    done, asked = False, None

    def record(self, stream=None):
        pass

    def synchronize(self):
        pass

    def query(self):
        if self.asked is not None:
            asked, self.asked = self.asked, None
            asked()
        time.sleep(0)
        return self.done


@pytest.fixture(autouse=True)
def stand_ins(monkeypatch):
    empty = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, pin_memory=False, **kw: empty(*a, **kw))
    monkeypatch.setattr(torch.cuda, "Event", Event)
    staging._retired.clear()
    yield
    staging._retired.clear()


def _sampler():
    """A sampler that has staged numbers once: itself, its event and a reference to its buffer."""
    s = S.Sampler(S.GenerationParams(seed=1))
    host, copied, _, _ = s._staging_buffer(10)
    return s, copied, weakref.ref(host)


def _end(holder):
    holder.clear()
    gc.collect()


def test_a_sampler_that_ends_while_another_ones_buffers_are_looked_at():
    a, b, c, d = ([_sampler()] for _ in range(4))
    kept = [x[0][2] for x in (a, b, c, d)]
    events = [x[0][1] for x in (a, b, c, d)]
    events[0].asked = lambda: _end(b)
    for x in (a, c, d):
        _end(x)
    rest = _sampler()                                       # (its buffer is a reason to look at the retired ones)
    assert all(k() is not None for k in kept) and not b
    for e in events:
        e.done = True
    rest[0]._staging_buffer(10)
    gc.collect()
    assert all(k() is None for k in kept) and not staging._retired


def test_samplers_that_end_on_several_threads():
    each, threads = 100, 4
    made = [[[_sampler()] for _ in range(each)] for _ in range(threads)]
    kept = [x[0][2] for xs in made for x in xs]
    events = [x[0][1] for xs in made for x in xs]
    keep_asking = _sampler()[0]
    start = threading.Barrier(threads)

    def end(xs):
        start.wait()
        for x in xs:
            x.clear()
            keep_asking._staging_buffer(10)
    interval = sys.getswitchinterval()
    sys.setswitchinterval(1e-6)
    try:
        workers = [threading.Thread(target=end, args=(xs,)) for xs in made]
        for w in workers:
            w.start()
        for w in workers:
            w.join(60)
    finally:
        sys.setswitchinterval(interval)
    assert not any(w.is_alive() for w in workers)
    assert sum(k() is not None for k in kept) == each * threads
    for e in events:
        e.done = True
    keep_asking._staging_buffer(10)
    gc.collect()
    assert sum(k() is not None for k in kept) == 0


def test_a_buffer_that_is_replaced_by_a_longer_one_waits_for_its_copy():
    s, copied, host = _sampler()
    for _ in range(4):
        s._staging_buffer(5000)                             # (the fourth is the first one's place)
    assert host() is not None and any(p[1] is copied for p in staging._retired)
    copied.done = True
    s._staging_buffer(5000)
    gc.collect()
    assert host() is None and not any(p[1] is copied for p in staging._retired)


def test_an_event_that_can_not_be_asked_keeps_its_buffer():
    a, rest = [_sampler()], _sampler()[0]
    kept, event = a[0][2], a[0][1]

    def fail():
        raise RuntimeError("busy")
    event.asked = fail
    _end(a)
    with pytest.raises(RuntimeError, match="busy"):
        rest._staging_buffer(10)
    gc.collect()
    assert kept() is not None


@pytest.mark.parametrize("current", [0, 1])
def test_logits_on_a_device_that_is_not_the_current_one(current, monkeypatch):
    """Everything that a draw queues is the logits' device's: an event is its first record's device's, and refuses another one's stream."""
    import contextlib
    from types import SimpleNamespace
    now = [current]

    class OnDevice(Event):
        device, cuda_event = None, 0

        def record(self, stream=None):
            at = now[0] if stream is None else stream
            self.device = at if self.device is None else self.device
            assert self.device == at, "the event's device is not the stream's"

    @contextlib.contextmanager
    def device(d):
        before, now[0] = now[0], d.index
        yield
        now[0] = before
    monkeypatch.setattr(torch.cuda, "Event", OnDevice)
    monkeypatch.setattr(torch.cuda, "device", device)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: now[0])
    monkeypatch.setattr(torch.cuda, "current_stream", lambda d=None: now[0] if d is None else d)
    drawn = []

    def draw(*a):
        drawn.append(now[0])
        return "ids"
    monkeypatch.setattr(staging, "K", SimpleNamespace(**{**vars(staging.K), "sample_few_serves": lambda *a: True, "sample_few_staged": draw}))

    class Logits:
        device, shape, is_cuda = SimpleNamespace(index=1, type="cuda"), (2, 100), True
        dim = staticmethod(lambda: 2)
        is_contiguous = staticmethod(lambda: True)
    s = S.Sampler(S.GenerationParams(seed=1, repetition_penalty=1.0))
    for step in range(6):
        assert s.sample(Logits(), [0, 1], [step, step]) == "ids"
    assert drawn == [1] * 6 and now == [current]
    assert all(p[1].device == 1 for p in s._staging.values())
