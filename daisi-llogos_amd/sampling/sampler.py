"""Token selection for a batch of logit rows, on the device.

The pipeline is the reference's (Daisi.Llogos/Inference/Sampler.cs:26-85): greedy short cut,
penalties, temperature, top-k, min-p, softmax over candidates, typical-p, top-p, draw."""
from __future__ import annotations

import struct
import weakref
from collections import deque
from typing import List, Optional, Sequence

import numpy as np
import torch

from ..ops import kernels as K, library
from .params import GenerationParams
from .rng import uniforms


# Staging buffers that nobody fills any more, until their last copies have run: those are queued by the kernel library, so that torch
# would hand freed pinned memory out again while one still reads it.  Samplers end on any thread, in the middle of anything (a collection of
# cycles): what ends only appends, and one buffer at a time is taken out, looked at and, if still needed, put back.
_retired: deque = deque()


def _retire(places: dict) -> None:
    for place in list(places.values()):
        _retired.append(place)


def _give_back() -> None:
    """Lets go of the retired buffers whose last copies have run."""
    for _ in range(len(_retired)):
        try:
            place = _retired.popleft()
        except IndexError:                          # (another thread was quicker)
            return
        done = False
        try:
            done = place[1].query()
        finally:
            if not done:
                _retired.append(place)


class Sampler:
    _settings = _settings_of = None         # as the kernels take them, and of which parameters and banned tokens they were made
    _staging, _staging_next = None, 0       # number -> staging buffer, its event, its bytes and its address; the number used last

    def __init__(self, params: GenerationParams, stop_tokens: Sequence[int] = ()):
        self.params = params
        self.stop_tokens = tuple(stop_tokens)
        if params.prevent_eos and len(self.stop_tokens) > K.MAX_BANNED:
            raise ValueError(f"prevent_eos can ban at most {K.MAX_BANNED} stop tokens, got {len(self.stop_tokens)}")
        self._fresh_seed = None
        if params.seed is None and params.temperature > 0:
            self._fresh_seed = int(np.random.SeedSequence().generate_state(1)[0])

    def uniforms(self, requests: Sequence[int], indices: Sequence[int]) -> List[float]:
        seed = self.params.seed if self.params.seed is not None else self._fresh_seed
        return uniforms(seed, requests, indices)

    def sample(self, logits: torch.Tensor, requests: Sequence[int], indices: Sequence[int],
               histories: Optional[Sequence[Sequence[int]]] = None) -> torch.Tensor:
        """int32 token ids [R] for float32 logits [R, V].  requests/indices: which request each
        row belongs to and which of its generated tokens this is (for the random stream);
        histories: each row's prompt + generated tokens (for penalties)."""
        if logits.is_cuda and logits.device.index != torch.cuda.current_device():
            with torch.cuda.device(logits.device):          # (kernels, copies and the staging buffers' events are all that device's)
                return self.sample(logits, requests, indices, histories)
        p = self.params
        if p.is_greedy:
            return K.argmax(logits)
        if p.has_penalties and histories is None:
            raise ValueError("penalties need each row's token history")
        if p.temperature > 0 and logits.dim() == 2 and logits.is_contiguous() and K.sample_few_serves(*logits.shape, p.top_k):
            return self._sample_few(logits, requests, indices, histories)
        arrays = []
        if p.has_penalties:
            win = [list(h[-p.penalty_count:]) if 0 < p.penalty_count < len(h) else list(h) for h in histories]
            width = max(1, max(len(w) for w in win))
            arr = np.zeros((len(win), width), dtype=np.int32)
            for i, w in enumerate(win):
                arr[i, :len(w)] = w
            arrays = [arr, np.asarray([len(w) for w in win], dtype=np.int32)]
        if p.temperature > 0:
            arrays.append(np.asarray(self.uniforms(requests, indices), dtype=np.float32))
        staged = self._to_device(arrays, logits.device)
        hist, hist_len = (staged[0], staged[1]) if p.has_penalties else (None, None)
        banned = self.stop_tokens if p.prevent_eos else ()
        work = K.sample_prepare(logits, hist, hist_len, p.repetition_penalty, p.frequency_penalty,
                                p.presence_penalty, p.temperature, p.penalize_newline, banned)
        if p.temperature == 0:
            return K.argmax(work)
        return K.sample_pipeline(work, staged[-1], p.top_k, p.top_p, p.min_p, p.typical_p, p.min_keep)

    def _sample_few(self, logits: torch.Tensor, requests, indices, histories) -> torch.Tensor:
        """The same for a small top-k, whose rows two kernels take from the logits to the token."""
        p = self.params
        R = logits.shape[0]
        # one copy: uniform numbers, then each window's place and the windows, packed straight into the staging buffer
        starts, n, host, copied = self._pack(R, requests, indices, histories) or self._pack_in_python(requests, indices, histories)
        if starts != (R, 2 * R + 1 if p.has_penalties else R + 1):
            raise K.KernelError(f"sample: {R} rows of logits need a uniform number and, with penalties, a token history each")
        banned = self.stop_tokens if p.prevent_eos else ()
        key = (p, banned)
        if self._settings_of != key:
            self._settings = K.sample_settings(p.repetition_penalty, p.frequency_penalty, p.presence_penalty, p.temperature, p.penalize_newline,
                                               banned, p.top_k, p.top_p, p.min_p, p.typical_p, p.min_keep)
            self._settings_of = key
        return K.sample_few_staged(logits, host.data_ptr(), n, p.has_penalties, self._settings, copied.cuda_event)

    def _pack(self, R: int, requests, indices, histories):
        """((where the windows' places begin, where the windows do), 32-bit numbers in all, staging buffer, its event) with R rows' uniform numbers and
        windows in the buffer; None for what the host's helpers leave to Python (anything but lists and tuples of plain integers)."""
        p, helpers = self.params, library.host()
        if helpers is None or getattr(self.uniforms, "__func__", None) is not Sampler.uniforms:      # (or the numbers come from elsewhere)
            return None
        count = p.penalty_count
        if not (p.has_penalties and -1 << 62 < count < 1 << 62):
            size = -1 if p.has_penalties else 0
        else:
            size = helpers.llogos_host_windows_size(histories, count)
        if size < 0:
            return None
        rows = R + 1 if p.has_penalties else 1
        host, copied, _, address = self._staging_buffer(R + rows + size)
        seed = p.seed if p.seed is not None else self._fresh_seed
        if helpers.llogos_host_uniforms(seed, requests, indices, R, address) != 0:
            return None
        if p.has_penalties and helpers.llogos_host_windows(histories, count, R, address + 4 * R, address + 4 * (R + rows), size) != size:
            return None
        return (R, R + rows), R + rows + size, host, copied

    def _pack_in_python(self, requests, indices, histories):
        p = self.params
        us = self.uniforms(requests, indices)
        flat, at = [], [0]
        if p.has_penalties:
            for h in histories:
                flat += h[-p.penalty_count:] if 0 < p.penalty_count < len(h) else h
                at.append(len(flat))
        n = len(us) + len(at) + len(flat)
        host, copied, numbers, _ = self._staging_buffer(n)
        try:
            struct.pack_into(f"={len(us)}f{len(at) + len(flat)}i", numbers, 0, *us, *at, *flat)
        except (struct.error, TypeError):                # (tokens that are no whole numbers: as numpy rounds them)
            view = np.frombuffer(numbers, dtype=np.int32)
            view[:len(us)] = np.asarray(us, dtype=np.float32).view(np.int32)
            view[len(us):len(us) + len(at)] = at
            view[len(us) + len(at):n] = flat
        return (len(us), len(us) + len(at)), n, host, copied

    def _staging_buffer(self, n: int):
        """A pinned buffer of at least n 32-bit numbers, the event to record behind its copy, its memory as bytes and its address: one of a
        few, each free again once its last copy has run."""
        if _retired:
            _give_back()
        at = self._staging_next = (self._staging_next + 1) % 4
        place = self._staging.get(at) if self._staging is not None else None
        if place is None or place[0].numel() < n:
            if self._staging is None:
                self._staging = {}
                weakref.finalize(self, _retire, self._staging)
            elif place is not None:
                _retire({at: place})
            host = torch.empty(max(1024, 2 * n), dtype=torch.int32, pin_memory=True)
            place = self._staging[at] = (host, torch.cuda.Event(), memoryview(host.numpy()).cast("B"), host.data_ptr())
            place[1].record()                                    # (an event has no handle before it is recorded once)
            return place
        place[1].synchronize()
        return place

    def _to_device(self, arrays, device) -> List[torch.Tensor]:
        """The step's small host arrays (int32 or float32) on the device with one copy, without
        the host waiting for the work already queued there (a copy from ordinary host memory
        would): through one of a few pinned staging buffers, each free again once its last copy
        has run."""
        if not arrays:
            return []
        n = sum(a.size for a in arrays)
        host, copied, _, _ = self._staging_buffer(n)
        flat = host.numpy()
        o = 0
        for a in arrays:
            flat[o:o + a.size] = a.reshape(-1).view(np.int32)          # float32 goes as its bits
            o += a.size
        dev = torch.empty(n, dtype=torch.int32, device=device)
        dev.copy_(host[:n], non_blocking=True)
        copied.record()
        out, o = [], 0
        for a in arrays:
            t = dev[o:o + a.size]
            out.append((t.view(torch.float32) if a.dtype == np.float32 else t).view(a.shape))
            o += a.size
        return out
