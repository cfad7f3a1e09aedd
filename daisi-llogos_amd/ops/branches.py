"""A step's second branch: a part's work that is queued on a stream of its own beside the caller's (inside a captured step
the two become branches of the graph), until both meet again.

    side = branches.fork(device, streams)       # None: no second branch here, do it on the caller's stream
    if side is not None:
        with branches.branch(side):
            a = ...
    b = ...
    branches.join(device, side)

A branch does not fork again: ending the capture of a step with a fork inside a fork has ended the process (a segmentation fault on
the host, before any replay).  And since the two branches run at the same time, memory that calls of one stream hand to one
another in turn (attention's scratch and counters) is there once for each: in_branch() says to which of the two a call belongs,
in a step that is launched, in the run before a capture and in the capture alike."""
from __future__ import annotations

import contextlib
import threading
from typing import Dict, Optional

import torch

_here = threading.local()


def in_branch() -> bool:
    """Whether the calling thread is queueing a second branch's work."""
    return getattr(_here, "on", False)


def fork(device: torch.device, streams: Dict[torch.device, "torch.cuda.Stream"]) -> Optional["torch.cuda.Stream"]:
    """The stream of `streams` for the device (made if need be), behind everything that the current stream holds; None inside a branch."""
    if in_branch():
        return None
    side = streams.get(device)
    if side is None:
        side = streams[device] = torch.cuda.Stream(device=device)
    side.wait_stream(torch.cuda.current_stream(device))
    return side


@contextlib.contextmanager
def branch(side: "torch.cuda.Stream"):
    """What is called inside is queued on `side`."""
    _here.on = True
    try:
        with torch.cuda.stream(side):
            yield
    finally:
        _here.on = False


def join(device: torch.device, side: Optional["torch.cuda.Stream"]) -> None:
    """The current stream goes on once `side` is through (nothing for None)."""
    if side is not None:
        torch.cuda.current_stream(device).wait_stream(side)
