"""The host's helpers that pack the sampler's lists give what the Python beside them gives, and leave alone what is not theirs."""
import importlib
import random

import numpy as np
import pytest

library = importlib.import_module("daisi-llogos_amd.ops.library")
rng = importlib.import_module("daisi-llogos_amd.sampling.rng")


@pytest.fixture(scope="module")
def helpers():
    found = library.host()
    if found is None:
        pytest.skip("no headers of Python or no compiler here")
    return found


def _windows(helpers, histories, count, rows=None, room=None):
    size = helpers.llogos_host_windows_size(histories, count)
    if size < 0:
        return size
    n = len(histories) if rows is None else rows
    starts, flat = np.full(n + 2, -7, np.int32), np.full(size + 1, -7, np.int32)
    code = helpers.llogos_host_windows(histories, count, n, starts.ctypes.data, flat.ctypes.data, size if room is None else room)
    assert starts[-1] == -7 and flat[-1] == -7                                  # nothing behind the rooms
    return code if code < 0 else (starts[:-1].tolist(), flat[:-1].tolist())


@pytest.mark.parametrize("count", [0, 1, 5, 64, -3, 1 << 40])
def test_windows(helpers, count):
    draw = random.Random(count)
    histories = [[draw.randrange(-2 ** 31, 2 ** 31) for _ in range(n)] for n in (0, 1, 4, 5, 6, 63, 64, 65, 200)]
    want = [h[-count:] if 0 < count < len(h) else h for h in histories]
    starts = np.concatenate([[0], np.cumsum([len(h) for h in want])]).tolist()
    for given in (histories, tuple(histories), [tuple(h) for h in histories]):
        assert _windows(helpers, given, count) == (starts, sum(want, []))
    assert _windows(helpers, [], count) == ([0], [])


def test_windows_that_are_left_to_python(helpers):
    for histories in (None, "ab", iter([[1]]), [[1], "ab"], [[1], np.array([1])], np.zeros((2, 2), int), {1: [1]}):
        assert helpers.llogos_host_windows_size(histories, 4) == -1
    for bad in (2 ** 31, -2 ** 31 - 1, 1 << 80, 1.0, True, np.int32(3), None, "1"):
        assert _windows(helpers, [[1, 2], [3, bad]], 4) == -1
        assert _windows(helpers, [[bad, 2, 3]], 2) == ([0, 2], [2, 3])          # outside of the window it is not read
    assert _windows(helpers, [[1, 2]], 4, rows=2) == -1 and _windows(helpers, [[1, 2], [3]], 4, room=2) == -1


@pytest.mark.parametrize("seed", [0, 7, -1, 2 ** 64 + 5, 1 << 100])
def test_uniform_numbers(helpers, seed):
    requests, indices = [0, 1, 5, 2 ** 31, -1, 2 ** 64 - 1, 1 << 70], [0, 3, 2 ** 40, 1, -5, 2 ** 63, 9]
    out = np.zeros(len(requests) + 1, np.float32)
    for pair in ((requests, indices), (tuple(requests), indices)):
        assert helpers.llogos_host_uniforms(seed, *pair, len(requests), out.ctypes.data) == 0
        assert out[:-1].tolist() == [rng.uniform(seed, r, i) for r, i in zip(requests, indices)] and out[-1] == 0
    for bad in ((requests[:-1], indices), (requests, indices[:-1]), (iter(requests), indices), (requests, np.arange(7)), ([1.0] * 7, indices), ([True] * 7, indices)):
        assert helpers.llogos_host_uniforms(seed, *bad, len(requests), out.ctypes.data) == -1
    assert helpers.llogos_host_uniforms(1.5, requests, indices, len(requests), out.ctypes.data) == -1


def test_sampler_packs_the_same_either_way(helpers):
    """_pack and _pack_in_python fill a buffer alike (without a GPU: ordinary memory in the staging buffer's place)."""
    llogos = importlib.import_module("daisi-llogos_amd")
    draw = random.Random(1)
    for penalty in (1.0, 1.2):
        s = llogos.Sampler(llogos.GenerationParams(temperature=0.7, top_k=40, repetition_penalty=penalty, seed=3))
        buffer = np.zeros(4000, np.int32)
        s._staging_buffer = lambda n: (buffer, None, memoryview(buffer).cast("B"), buffer.ctypes.data)
        histories = [[draw.randrange(50000) for _ in range(draw.randrange(0, 150))] for _ in range(9)]
        requests, indices = list(range(9)), [draw.randrange(99) for _ in range(9)]
        buffer[:] = 0
        starts, n, _, _ = s._pack(9, requests, indices, histories)
        native = buffer.copy()
        buffer[:] = 0
        assert s._pack_in_python(requests, indices, histories)[:2] == (starts, n) and (buffer == native).all()
        assert s._pack(9, requests, indices[:-1], histories) is None and s._pack(9, map(int, requests), indices, histories) is None
