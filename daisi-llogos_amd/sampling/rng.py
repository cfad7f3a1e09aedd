"""Uniform numbers for sampling that depend on (seed, request, token index) alone, so a
request draws the same numbers whatever else is in its batch.  The reference draws from one
System.Random per sampler (Daisi.Llogos/Inference/Sampler.cs:12-15, 336); with one sequence
per sampler that is the same property."""
from __future__ import annotations

from typing import Iterable, List

import numpy as np

_MASK = (1 << 64) - 1


def _splitmix64(x: int) -> int:
    x = (x + 0x9E3779B97F4A7C15) & _MASK
    z = x
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & _MASK
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & _MASK
    return z ^ (z >> 31)


def uniform(seed: int, request: int, index: int) -> float:
    """A float32-exact number in [0, 1): 24 random bits."""
    h = _splitmix64(seed & _MASK)
    h = _splitmix64(h ^ ((request + 1) * 0xD6E8FEB86659FD93 & _MASK))
    h = _splitmix64(h ^ ((index + 1) * 0xA0761D6478BD642F & _MASK))
    return (h >> 40) / float(1 << 24)


def _splitmix64_array(x: np.ndarray) -> np.ndarray:
    z = x + np.uint64(0x9E3779B97F4A7C15)
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


def uniforms(seed: int, requests: Iterable[int], indices: Iterable[int]) -> List[float]:
    """uniform(seed, r, i) of each pair; from a few pairs on in arrays of 64-bit numbers, which wrap as the masks above do."""
    if not (isinstance(requests, (list, tuple)) and isinstance(indices, (list, tuple))):
        pairs = list(zip(requests, indices))                # (iterators and views have no length or no slices; one may be endless)
        requests, indices = [r for r, _ in pairs], [i for _, i in pairs]
    n = min(len(requests), len(indices))
    if n > 8:
        r, i = np.array(requests[:n]), np.array(indices[:n])
        if r.dtype.kind in "iu" and i.dtype.kind in "iu" and r.ndim == i.ndim == 1:
            h = np.uint64(_splitmix64(seed & _MASK))
            h = _splitmix64_array(h ^ (r.astype(np.uint64) + np.uint64(1)) * np.uint64(0xD6E8FEB86659FD93))
            h = _splitmix64_array(h ^ (i.astype(np.uint64) + np.uint64(1)) * np.uint64(0xA0761D6478BD642F))
            return ((h >> np.uint64(40)).astype(np.float64) / float(1 << 24)).tolist()
    return [uniform(seed, r, i) for r, i in zip(requests, indices)]
